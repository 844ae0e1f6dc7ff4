// One row of scores -> pyramid levels: the device code shared by the level-map kernel and the fused estimator
// epilogue, and the host-side parameter set-up.  See psa_level_map.hip for the algorithm.
#pragma once
#include "psa_common.h"

struct LevelMapParams {
  const float* scores;
  void* map_out;
  int32_t* list_out;
  int map_elem;
  int Nk;
  int mode;
  int n_items;
  int level[PSA_MAX_LEVEL_ITEMS];
  int align[PSA_MAX_LEVEL_ITEMS];
  float thr[PSA_MAX_LEVEL_ITEMS];     // thresholdbound: fp32(hi + 1e-6)
  int fixed_s[PSA_MAX_LEVEL_ITEMS];   // topk: row-independent intervals
  int fixed_e[PSA_MAX_LEVEL_ITEMS];
  // topk: the same intervals as cuts of the rank axis: ranks cut[s - 1] .. cut[s] - 1 get seg_level[s] (cut[-1] = 0)
  int n_cuts;
  int cut[2 * PSA_MAX_LEVEL_ITEMS];
  int seg_level[2 * PSA_MAX_LEVEL_ITEMS + 1];
  int min_index;                      // thresholdbound: floor for the level-1 interval
  int text_blocks;
};

__device__ __forceinline__ uint32_t desc_key(float s) {
  s += 0.0f;  // -0.0 -> +0.0 so that both zeros tie
  uint32_t u = __builtin_bit_cast(uint32_t, s);
  u ^= (u >> 31) ? 0xffffffffu : 0x80000000u;  // ascending order-preserving
  return ~u;                                   // descending
}

// Stable descending order of one row of scores: sidx[i] = column of sorted position i, sw[i] its score.
// The 64-bit keys (inverted score bits, column) are unique, so every correct sort gives the same order.
// Rows of up to RANK_SORT_MAX scores are ranked by counting (one pass of N comparisons per score, no barriers inside).  Longer ones are
// dealt to SORT_BINS bins, equal steps of the score bits between the row's best and worst (8 bins per octave for scores that reach from 1 down to
// the smallest floats, more otherwise), and ranked by counting inside their bin: a few comparisons per score and six barriers.
// A bin of more than SORT_TIES scores is mostly scores equal to the worst (the zeros above a causal diagonal, scores that underflow,
// rows that are all alike): those are placed in column order, by ballots, and their bin is ranked without them.  If a bin of a row of more than 256
// still has more than SORT_CAP (scores of a few values), the row goes through a bitonic network over key[0 .. sort_pad).
// Against ranking up to 256 scores by counting and longer rows by the network, reduction + map of estimates by attention mass, us: 40 heads x
// 10750 tokens of 32-key blocks (336 scores) 102 -> 66, 24 x 13273 (415) 73 -> 53, 12 x 32760 of 128-key blocks (256) 58 -> 46.  Maps alone, us,
// then / now, continuous scores and rows of which 84 % are 0: 8192 rows of 129 scores 42 / 39, 42 / 43; of 256 73 / 55, 73 / 61; of 512
// 149 / 98, 148 / 109; 4096 of 1024 161 / 105, 159 / 115; 1024 of 4096 564 / 360, 562 / 350.  Causal maps of their own (28 heads of
// 200 x 200, zeros above the diagonal) 39 / 33.  (Without the placing of ties: 67, 90, 156, 171, 592, and 50.)  Rows of nine values pay for the
// bins in vain: 129 scores 42 / 53, 256 73 / 83, 4096 564 / 599.
constexpr int RANK_SORT_MAX = 128, SORT_BINS = 1024, SORT_TIES = 32, SORT_CAP = 128;
__host__ __device__ inline int sort_pad(int N) {
  if (N <= RANK_SORT_MAX) return N;
  int n = 1;
  while (n < N) n <<= 1;
  return n;
}
// LDS, in words of 4 bytes: [hist, later the prefix sums: sort_hist(N)][keys: 2 * sort_pad(N)][sw: N][sidx: N].  Rows longer than
// RANK_SORT_MAX: 256 threads.
__host__ __device__ inline int sort_hist(int N) {
  const int n = (N + 3) & ~3;  // (the histogram and the keys behind it are read 16 bytes at a time)
  return N > RANK_SORT_MAX && n < SORT_BINS ? SORT_BINS : n;
}
__host__ __device__ inline size_t sort_lds_bytes(int N) { return (size_t)sort_hist(N) * 4 + (size_t)sort_pad(N) * 8 + (size_t)N * 8; }
__device__ __forceinline__ void sort_row_desc(uint64_t* key, float* sw, int* sidx, uint32_t* hist, const float* src, int N, int tid, int nt) {
  if (N <= RANK_SORT_MAX) {
    for (int j = tid; j < N; j += nt) key[j] = ((uint64_t)desc_key(src[j]) << 32) | (uint32_t)j;
    __syncthreads();
    for (int j = tid; j < N; j += nt) {
      const uint64_t kj = key[j];
      int rank = 0;
      for (int i = 0; i < N; ++i) rank += key[i] < kj ? 1 : 0;
      sw[rank] = src[j];
      sidx[rank] = j;
    }
    __syncthreads();
    return;
  }
  constexpr int NT = 256, NW = NT / 64;
  static_assert(SORT_BINS == 4 * NT, "a thread scans four bins");
  __shared__ uint32_t s_lo[NW], s_hi[NW], s_sum[NW], s_most[NW];
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  ((u32x4*)hist)[tid] = u32x4{0u, 0u, 0u, 0u};
  uint32_t* kbuf = (uint32_t*)sidx;  // (the score bits, until the columns take their place)
  uint32_t lo = 0xffffffffu, hi = 0u;
  for (int j = tid; j < N; j += NT) {
    const uint32_t k = desc_key(src[j]);
    kbuf[j] = k;
    lo = k < lo ? k : lo;
    hi = k > hi ? k : hi;
  }
  lo = wave_min_u32(lo);
  hi = wave_max_u32(hi);
  if (lane == 0) {
    s_lo[wave] = lo;
    s_hi[wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    lo = s_lo[w] < lo ? s_lo[w] : lo;
    hi = s_hi[w] > hi ? s_hi[w] : hi;
  }
  const int bits = 32 - __builtin_clz((hi - lo) | 1u), shift = bits > 10 ? bits - 10 : 0;
  bool ties = false;                                       // many columns have the worst score: they are placed in column order
  const int span = ((N + NT - 1) / NT) * 64, c0 = wave * span, c1 = c0 + span < N ? c0 + span : N;  // columns of this wave where there are
  uint32_t at = 0;                                         // ... and where its tied ones go
  static_assert(SORT_BINS == 1 << 10, "bins");
  for (int j = tid; j < N; j += NT) atomicAdd(&hist[(kbuf[j] - lo) >> shift], 1u);
  __syncthreads();
  {
    u32x4 c = ((const u32x4*)hist)[tid];
    const uint32_t sum = c[0] + c[1] + c[2] + c[3];
    uint32_t most = c[0] > c[1] ? c[0] : c[1];
    most = c[2] > most ? c[2] : most;
    most = wave_max_u32(c[3] > most ? c[3] : most);
    uint32_t run = (uint32_t)wave_scan_add((int)sum);
    if (lane == 63) s_sum[wave] = run;
    if (lane == 0) s_most[wave] = most;
    run -= sum;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) run += w < wave ? s_sum[w] : 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t n = c[e];
      c[e] = run;
      run += n;
    }
    ((u32x4*)hist)[tid] = c;
    most = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) most = s_most[w] > most ? s_most[w] : most;
    if (most > (uint32_t)SORT_TIES) {  // (uniform)
      uint32_t n = 0;
      for (int j0 = c0; j0 < c1; j0 += 64) n += (uint32_t)__popcll(__ballot(j0 + lane < c1 && kbuf[j0 + lane < c1 ? j0 + lane : 0] == hi));
      if (lane == 0) s_lo[wave] = n;
      __syncthreads();
      const uint32_t tied = s_lo[0] + s_lo[1] + s_lo[2] + s_lo[3];
      ties = tied > 1;
      at = (uint32_t)N;
#pragma unroll
      for (int w = 0; w < NW; ++w) at -= w >= wave ? s_lo[w] : 0u;
      if (N > 256 && most > (uint32_t)SORT_CAP) {  // without the tied columns, which are at the end of the last bin
        most = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t in = (e < 3 ? c[e < 3 ? e + 1 : 3] : run) - c[e];
          in -= (uint32_t)(4 * tid + e) == (hi - lo) >> shift ? tied : 0u;
          most = in > most ? in : most;
        }
        most = wave_max_u32(most);
        if (lane == 0) s_hi[wave] = most;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; ++w) most = s_hi[w] > most ? s_hi[w] : most;
        if (most > (uint32_t)SORT_CAP) {
          const int Npad = sort_pad(N);
          for (int j = tid; j < Npad; j += NT) key[j] = j < N ? (((uint64_t)kbuf[j] << 32) | (uint32_t)j) : ~0ull;
          __syncthreads();
          for (int k = 2; k <= Npad; k <<= 1) {
            for (int j = k >> 1; j > 0; j >>= 1) {
              for (int e = tid; e < (Npad >> 1); e += NT) {
                // pair e of this stage: i has bit j clear, its partner is i + j; ascending where bit k of i is clear
                const int i = ((e & ~(j - 1)) << 1) | (e & (j - 1));
                const uint64_t a = key[i], b = key[i + j];
                const bool up = (i & k) == 0;
                if ((a > b) == up) {
                  key[i] = b;
                  key[i + j] = a;
                }
              }
              __syncthreads();
            }
          }
          for (int i = tid; i < N; i += NT) {
            const int col = (int)(uint32_t)key[i];
            sidx[i] = col;
            sw[i] = src[col];
          }
          __syncthreads();
          return;
        }
      }
    }
  }
  __syncthreads();
  // hist[b]: the next free place of bin b, in the end the first place of bin b + 1
  if (ties) {
    for (int j0 = c0; j0 < c1; j0 += 64) {
      const int j = j0 + lane;
      const uint32_t k = kbuf[j < c1 ? j : 0];
      const uint64_t tied = __ballot(j < c1 && k == hi);
      if (j < c1) {
        const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(tied >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)tied, 0u));
        key[k == hi ? at + before : atomicAdd(&hist[(k - lo) >> shift], 1u)] = ((uint64_t)k << 32) | (uint32_t)j;
      }
      at += (uint32_t)__popcll(tied);
    }
  } else {
    for (int j = tid; j < N; j += NT) {
      const uint32_t k = kbuf[j];
      key[atomicAdd(&hist[(k - lo) >> shift], 1u)] = ((uint64_t)k << 32) | (uint32_t)j;
    }
  }
  __syncthreads();
  for (int i = tid; i < N; i += NT) {
    const uint64_t mine = key[i];
    const uint32_t k = (uint32_t)(mine >> 32), bin = (k - lo) >> shift;
    int rank = i;
    if (!ties || k != hi) {
      const int first = bin > 0 ? (int)hist[bin - 1] : 0, last = (int)hist[bin];
      rank = first;
      for (int e = first; e < last; ++e) rank += key[e] < mine ? 1 : 0;
    }
    const int col = (int)(uint32_t)mine;
    sidx[rank] = col;
    sw[rank] = src[col];
  }
  __syncthreads();
}

// Prefix sums of the sorted scores, accumulated strictly sequentially in fp64 and rounded to fp32 (the order
// matters for bit-exactness).  All threads widen the scores into `wide` (the sort's key buffer, free by now) and
// round the sums afterwards, so that the dependent chain one lane has to run is a load, an addition and a store
// per two scores; that lane runs it at raised wave priority, because up to seven other waves compete with it for
// every instruction slot of the SIMD and the rest of its workgroup waits for it.
__device__ __forceinline__ void row_prefix_sums(double* wide, const float* sw, float* c32, int N, int tid, int nt) {
  typedef double f64x2 __attribute__((ext_vector_type(2)));
  for (int i = tid; i < N; i += nt) wide[i] = (double)sw[i];
  __syncthreads();
  if (tid == 0) {
    __builtin_amdgcn_s_setprio(3);
    double acc = 0.0;
    // eight scores at a time, the next eight requested before they are added: the chain is the additions, not the LDS
    f64x2 w[4], nx[4];
    const int n8 = N & ~7;
    if (n8 > 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) nx[e] = *(const f64x2*)(wide + 2 * e);
    }
    int i = 0;
    for (; i < n8; i += 8) {
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = nx[e];
      const int at = i + 8 < n8 ? i + 8 : i;  // (the last one's repeat is not used)
#pragma unroll
      for (int e = 0; e < 4; ++e) nx[e] = *(const f64x2*)(wide + at + 2 * e);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[e][0] = acc + w[e][0];
        w[e][1] = acc = w[e][0] + w[e][1];
        *(f64x2*)(wide + i + 2 * e) = w[e];
      }
    }
    for (; i < N; ++i) {
      acc += wide[i];
      wide[i] = acc;
    }
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();
  for (int i = tid; i < N; i += nt) c32[i] = (float)wide[i];
  __syncthreads();
}

// Levels by fixed quotas need no sorted row: the level of a column follows from how many of the `n_cuts` keys of rank
// cut[0], cut[1], .. its own key reaches.  A histogram of the keys (SEL_BINS bins, 16 per octave below the row's best
// score) finds the bin of every cut, the few keys in that bin are ranked by counting, and one pass compares each key
// with the cut keys.  A cut whose bin holds more than SEL_CAP keys descends into it: a histogram of the bin's (key, column)
// range in SEL_BINS finer bins, until the cut's bin fits.  One descent is enough for flat rows (logits of standard deviation 0.25
// to 1 put one to three cuts of a row of 512 to 2048 scores there), equal scores take up to three more, down to the column.
// Bound by latency (a dozen barriers, six more per descent).  3072 rows of 1024 scores in us, logits of deviation 3 / 1 / 0.5 /
// 0.25: 21 / 26 / 34 / 41, bitonic network 65 to 71 whatever the scores; 3072 rows of 512: 17 / 18 / 20 / 28 against 34; of
// 2048: 31 / 46 / 58 / 60 against 200.  (Building the cut key bit by bit over the whole row instead of descending: 21 / 58 / 138 /
// 266 at 1024 scores.)  With the reduction of the estimator's workspace, which the launch also does and which bounds it: 16944
// rows of 1410 scores 1480 -> 600 us (3.05 GB read, 5.1 TB/s).  Up to SEL_MIN scores sorting is as fast and also
// serves the other modes.
// LDS: (SEL_BINS + 2 * SEL_MAX_CUTS * SEL_CAP + 8 * SEL_MAX_CUTS) 4-byte words.  256 threads.
constexpr int SEL_MIN = 256, SEL_BINS = 1024, SEL_SHIFT = 19, SEL_CAP = 64, SEL_MAX_CUTS = 8;
constexpr int SEL_COL_BITS = 13;  // columns of a row: at most 6144
constexpr size_t SEL_LDS_BYTES = (SEL_BINS + 2 * SEL_MAX_CUTS * SEL_CAP + 8 * SEL_MAX_CUTS) * 4;
__host__ __device__ inline bool level_map_selects(int mode, int n_cuts, int Nk) {
  return mode == PSA_MODE_TOPK && n_cuts <= SEL_MAX_CUTS && Nk > SEL_MIN;
}
__device__ __forceinline__ void level_map_row_select(const LevelMapParams& p, const float* src, int64_t row, unsigned char* smem, int tid,
                                                     uint8_t* lds_out) {
  constexpr int NT = 256, PER = SEL_BINS / NT;
  uint64_t* cand = (uint64_t*)smem;                       // [cut][SEL_CAP] keys of the bin that holds the cut
  uint64_t* cut_key = cand + SEL_MAX_CUTS * SEL_CAP;      // [cut] key of rank cut[c]
  int* hist = (int*)(cut_key + SEL_MAX_CUTS);             // [SEL_BINS]
  int* bin_of = hist + SEL_BINS;                          // [cut] bin that holds the cut
  int* before = bin_of + SEL_MAX_CUTS;                    // [cut] keys in earlier bins
  int* n_in = before + SEL_MAX_CUTS;                      // [cut] keys in that bin
  int* fill = n_in + SEL_MAX_CUTS;                        // [cut] keys collected so far
  int* wsum = fill + SEL_MAX_CUTS;                        // [8] partial results of the waves
  int* found = wsum + 8;                                  // [3] bin of a cut inside a crowded bin, keys before it, keys in it
  const int N = p.Nk, lane = tid & 63, wave = tid >> 6, C = p.n_cuts;

  for (int i = tid; i < SEL_BINS; i += NT) hist[i] = 0;
  if (tid < SEL_MAX_CUTS) fill[tid] = 0;
  uint32_t kmin = 0xffffffffu;
  for (int j = tid; j < N; j += NT) {
    const uint32_t k = desc_key(src[j]);
    kmin = k < kmin ? k : kmin;
  }
  kmin = wave_min_u32(kmin);
  if (lane == 0) wsum[wave] = (int)kmin;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const uint32_t k = (uint32_t)wsum[w];
    kmin = k < kmin ? k : kmin;
  }
  auto bin_at = [&](uint32_t k) __attribute__((always_inline)) {
    const uint32_t b = (k - kmin) >> SEL_SHIFT;
    return (int)(b < SEL_BINS - 1 ? b : SEL_BINS - 1);
  };
  for (int j = tid; j < N; j += NT) atomicAdd(&hist[bin_at(desc_key(src[j]))], 1);
  __syncthreads();
  // hit(bin, keys before it, keys in it) for every bin that holds keys (one barrier inside)
  auto scan_hist = [&](auto hit) __attribute__((always_inline)) {
    int c[PER], sum = 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      c[e] = hist[tid * PER + e];
      sum += c[e];
    }
    const int incl = wave_scan_add(sum);
    if (lane == 63) wsum[4 + wave] = incl;
    __syncthreads();
    int run = incl - sum;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) run += w < wave ? wsum[4 + w] : 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      if (c[e] > 0) hit(tid * PER + e, run, c[e]);
      run += c[e];
    }
  };
  scan_hist([&](int bin, int first, int n) __attribute__((always_inline)) {
    for (int t = 0; t < C; ++t)
      if (p.cut[t] >= first && p.cut[t] < first + n) {
        bin_of[t] = bin;
        before[t] = first;
        n_in[t] = n;
      }
  });
  __syncthreads();
  int cut_bin[SEL_MAX_CUTS];
#pragma unroll
  for (int t = 0; t < SEL_MAX_CUTS; ++t) cut_bin[t] = t < C ? bin_of[t] : -1;
  for (int j = tid; j < N; j += NT) {
    const uint32_t k = desc_key(src[j]);
    const int b = bin_at(k);
#pragma unroll
    for (int t = 0; t < SEL_MAX_CUTS; ++t)
      if (b == cut_bin[t]) {
        const int at = atomicAdd(&fill[t], 1);
        if (at < SEL_CAP) cand[t * SEL_CAP + at] = ((uint64_t)k << 32) | (uint32_t)j;
      }
  }
  __syncthreads();
  // the key of rank `rank` among the n candidates of cut t (one wave)
  auto rank_cand = [&](int t, int n, int rank) __attribute__((always_inline)) {
    const uint64_t mine = lane < n ? cand[t * SEL_CAP + lane] : ~0ull;
    int below = 0;
    for (int i = 0; i < n; ++i) below += cand[t * SEL_CAP + i] < mine ? 1 : 0;
    if (lane < n && below == rank) cut_key[t] = mine;
  };
  bool crowded = false;
#pragma unroll
  for (int t = 0; t < SEL_MAX_CUTS; ++t)
    if (t < C) {
      const int n = n_in[t];
      if (n > SEL_CAP) {
        crowded = true;
      } else if ((t & 3) == wave) {
        rank_cand(t, n, p.cut[t] - before[t]);
      }
    }
  if (crowded) {  // uniform: the counts are the same for every thread
    for (int t = 0; t < C; ++t) {
      int n = n_in[t], rank = p.cut[t] - before[t];
      if (n <= SEL_CAP) continue;
      // the cut's bin as a range of (score key, column), 2^bits wide from lo (the last bin: everything past its start)
      int bits = bin_of[t] < SEL_BINS - 1 ? SEL_SHIFT + SEL_COL_BITS : 32 + SEL_COL_BITS;
      uint64_t lo = (uint64_t)(kmin + ((uint32_t)bin_of[t] << SEL_SHIFT)) << SEL_COL_BITS;
      auto offset = [&](int j) __attribute__((always_inline)) { return (((uint64_t)desc_key(src[j]) << SEL_COL_BITS) | (uint32_t)j) - lo; };
      while (n > SEL_CAP) {  // (keys are unique: 64 of them span more than 5 bits)
        const int shift = bits - 10;
        for (int i = tid; i < SEL_BINS; i += NT) hist[i] = 0;
        __syncthreads();
        for (int j = tid; j < N; j += NT) {
          const uint64_t d = offset(j);
          if (d >> bits == 0) atomicAdd(&hist[(int)(d >> shift)], 1);
        }
        __syncthreads();
        scan_hist([&](int bin, int first, int cnt) __attribute__((always_inline)) {
          if (rank >= first && rank < first + cnt) {
            found[0] = bin;
            found[1] = first;
            found[2] = cnt;
          }
        });
        __syncthreads();
        lo += (uint64_t)(uint32_t)found[0] << shift;
        rank -= found[1];
        n = found[2];
        bits = shift;
      }
      if (tid == 0) fill[t] = 0;
      __syncthreads();
      for (int j = tid; j < N; j += NT)
        if (offset(j) >> bits == 0) cand[t * SEL_CAP + atomicAdd(&fill[t], 1)] = ((uint64_t)desc_key(src[j]) << 32) | (uint32_t)j;
      __syncthreads();
      if ((t & 3) == wave) rank_cand(t, n, rank);
    }
  }
  __syncthreads();
  uint64_t ck[SEL_MAX_CUTS];
#pragma unroll
  for (int t = 0; t < SEL_MAX_CUTS; ++t) ck[t] = t < C ? cut_key[t] : ~0ull;
  for (int j = tid; j < N; j += NT) {
    const uint64_t k = ((uint64_t)desc_key(src[j]) << 32) | (uint32_t)j;
    int lv = p.seg_level[0];
#pragma unroll
    for (int t = 0; t < SEL_MAX_CUTS; ++t) lv = k >= ck[t] ? p.seg_level[t + 1] : lv;
    if (j >= N - p.text_blocks) lv = 1;
    if (lds_out != nullptr) lds_out[j] = (uint8_t)lv;
    else store_map(p.map_out, row * N + j, p.map_elem, lv);
  }
}

// One row of the level map.  `src` = the row's N scores (global memory or LDS), `smem` = level_map_lds_bytes(p) bytes
// of 16-byte aligned LDS, s_cnt / s_iv = PSA_MAX_LEVEL_ITEMS (x2) ints of LDS; called by all nt threads of the workgroup.
// lds_out: the levels go there (a byte per column, LDS) instead of to p.map_out.
__device__ __forceinline__ void level_map_row(const LevelMapParams& p, const float* src, int64_t row, unsigned char* smem,
                                              int* s_cnt, int (*s_iv)[2], int tid, int nt, uint8_t* lds_out = nullptr) {
  const int N = p.Nk;
  if (p.list_out == nullptr && level_map_selects(p.mode, p.n_cuts, N)) {
    level_map_row_select(p, src, row, smem, tid, lds_out);
    return;
  }
  uint32_t* hist = (uint32_t*)smem;           // [sort_hist(N)]
  float* c32 = (float*)hist;                  // [N] prefix sums
  uint64_t* key = (uint64_t*)(hist + sort_hist(N));  // [sort_pad(N)]
  float* sw = (float*)(key + sort_pad(N));    // [N] scores in sorted order
  int* sidx = (int*)(sw + N);                 // [N] column of sorted position

  if (tid < PSA_MAX_LEVEL_ITEMS) s_cnt[tid] = 0;
  sort_row_desc(key, sw, sidx, hist, src, N, tid, nt);

  if (p.mode == PSA_MODE_THRESHOLDBOUND) {
    row_prefix_sums((double*)key, sw, c32, N, tid, nt);
    const float total = c32[N - 1];
    // positions whose cumulative ratio is within each item's bound: one ballot per item and pass, one LDS
    // atomic per wave and item (integer counts: the order of the additions does not matter)
    int local[PSA_MAX_LEVEL_ITEMS];
#pragma unroll
    for (int t = 0; t < PSA_MAX_LEVEL_ITEMS; ++t) local[t] = 0;
    for (int i0 = 0; i0 < N; i0 += nt) {
      const int i = i0 + tid;
      const float r = i < N ? c32[i] / total : 0.f;
#pragma unroll
      for (int t = 0; t < PSA_MAX_LEVEL_ITEMS; ++t)
        if (t < p.n_items) local[t] += __popcll(__ballot(i < N && r <= p.thr[t]));
    }
    if ((tid & 63) == 0) {
#pragma unroll
      for (int t = 0; t < PSA_MAX_LEVEL_ITEMS; ++t)
        if (t < p.n_items && local[t]) atomicAdd(&s_cnt[t], local[t]);
    }
    __syncthreads();
    if (tid == 0) {
      // a short dependent chain in one lane while the workgroup waits: raised priority, and no integer
      // division for the usual power-of-two alignments
      __builtin_amdgcn_s_setprio(3);
      int last = 0;
      for (int t = 0; t < p.n_items; ++t) {
        const int cnt = s_cnt[t];
        const int end0 = cnt > 0 ? cnt + 1 : last;
        const int start = last;
        const int al = p.align[t];
        int end;
        if (al > 1) {
          int len = end0 - start;
          len = len > 0 ? len : 0;
          const bool pow2 = (al & (al - 1)) == 0;
          const int rem = pow2 ? (len & (al - 1)) : len % al;
          if (rem) len += al - rem;
          end = start + len;
          end = end < N ? end : N;
          if (end == N) end = start + (pow2 ? ((end - start) & ~(al - 1)) : ((end - start) / al) * al);
        } else {
          end = end0 < 0 ? 0 : (end0 > N ? N : end0);
          end = end > start ? end : start;
          if (p.level[t] == 1) end = end > p.min_index ? end : p.min_index;
        }
        s_iv[t][0] = start;
        s_iv[t][1] = end;
        last = end;
      }
      __builtin_amdgcn_s_setprio(0);
    }
  } else {
    if (tid < p.n_items) {
      s_iv[tid][0] = p.fixed_s[tid];
      s_iv[tid][1] = p.fixed_e[tid];
    }
  }
  __syncthreads();

  if (p.map_out) {
    for (int i = tid; i < N; i += nt) {
      int lv = 0;
      for (int t = 0; t < p.n_items; ++t)
        if (i >= s_iv[t][0] && i < s_iv[t][1]) lv = p.level[t];
      const int col = sidx[i];
      if (col >= N - p.text_blocks) lv = 1;
      if (lds_out != nullptr) lds_out[col] = (uint8_t)lv;
      else store_map(p.map_out, row * N + col, p.map_elem, lv);
    }
  }
  if (p.list_out) {
    const int W = N + p.n_items;
    int32_t* dst = p.list_out + row * W;
    for (int cidx = tid; cidx < W; cidx += nt) {
      int v = 0;
      for (int t = 0; t < p.n_items; ++t) {
        const int pos = cidx - t;  // sorted position if this column belongs to segment t
        if (pos >= s_iv[t][0] && pos < s_iv[t][1]) v = sidx[pos];
        int sep = s_iv[t][1] + t;
        sep = sep > W - 1 ? W - 1 : sep;
        if (cidx == sep) v = -1;   // a separator written for item t survives later items' segments
      }
      dst[cidx] = v;
    }
  }
}


// ---- the causal Qwen2.5-VL example: square map, per-row ratio windows, fix-ups (psa_level_map.hip) ----
struct QwenMapParams {
  const float* scores;
  void* map_out;
  int map_elem;
  int S;       // blocks per side
  int mode;    // PSA_MODE_TOPK: rank windows on the causal row length; PSA_MODE_THRESHOLDBOUND: cumulative-mass windows
  int n_items;
  int level[PSA_MAX_LEVEL_ITEMS];
  float lo[PSA_MAX_LEVEL_ITEMS];  // energy mode: max(lo, previous hi); rank mode: lo
  float hi[PSA_MAX_LEVEL_ITEMS];
  int special;  // trailing blocks (rows and columns) forced to level 1
  int causal;
};
// LDS of a row of n scores
__host__ __device__ inline size_t qwen_row_lds_bytes(int n) { return sort_lds_bytes(n); }
// Levels of row i_row from its scores `src`, handed to store(column, level).  Only the first n columns are ranked: n = S, or the
// i_row + 1 columns of a causal row whose other scores are all 0 - those sort last whatever the rest (no score is negative), add
// nothing to a prefix sum and are skipped above the diagonal anyway.
template <class Store>
__device__ __forceinline__ void qwen_map_row(const QwenMapParams& p, const float* src, int i_row, int n, unsigned char* smem, int tid, int nt,
                                             Store store) {
  uint32_t* hist = (uint32_t*)smem;
  float* c32 = (float*)hist;
  uint64_t* key = (uint64_t*)(hist + sort_hist(n));
  float* sw = (float*)(key + sort_pad(n));
  int* sidx = (int*)(sw + n);
  sort_row_desc(key, sw, sidx, hist, src, n, tid, nt);
  if (p.mode == PSA_MODE_THRESHOLDBOUND) row_prefix_sums((double*)key, sw, c32, n, tid, nt);
  const float total = p.mode == PSA_MODE_THRESHOLDBOUND ? fmaxf(c32[n - 1], 1e-10f) : 1.f;
  const float valid_len = p.causal ? (float)(i_row + 1) : (float)p.S;
  for (int pos = tid; pos < n; pos += nt) {
    int lv = 0;
    if (p.mode == PSA_MODE_THRESHOLDBOUND) {
      const float r = c32[pos] / total;
      for (int t = 0; t < p.n_items; ++t)
        if (r > p.lo[t] && r <= p.hi[t]) lv = p.level[t];
    } else {
      for (int t = 0; t < p.n_items; ++t) {
        int s0 = (int)(valid_len * p.lo[t]), e0 = (int)(valid_len * p.hi[t]);
        s0 = s0 < p.S ? s0 : p.S;
        e0 = e0 < p.S ? e0 : p.S;
        if (pos >= s0 && pos < e0) lv = p.level[t];
      }
    }
    const int col = sidx[pos];
    if (col >= p.S - p.special || i_row >= p.S - p.special) lv = 1;
    if (p.causal && col > i_row) lv = 0;
    if (col == i_row || col == 0) lv = 1;
    store(col, lv);
  }
  for (int col = n + tid; col < p.S; col += nt) store(col, 0);  // (n < S: above the diagonal)
}

static inline int qwen_map_fill_params(QwenMapParams& p, int S, int mode, int n_items, const int32_t* item_level, const double* item_lo,
                                       const double* item_hi, int special_blocks, int causal) {
  PSA_REQUIRE(item_level && item_lo && item_hi, PSA_ERR_ARG, "psa_level_map_qwen: null pointer");
  PSA_REQUIRE(mode == PSA_MODE_TOPK || mode == PSA_MODE_THRESHOLDBOUND, PSA_ERR_ARG, "mode must be 'topk' or 'energybound'");
  PSA_REQUIRE(n_items >= 1 && n_items <= PSA_MAX_LEVEL_ITEMS, PSA_ERR_ARG, "mask_ratios must not be empty (1..%d items)", PSA_MAX_LEVEL_ITEMS);
  PSA_REQUIRE(S > 0 && S <= 6144, PSA_ERR_UNSUPPORTED, "psa_level_map_qwen: sizes out of range");
  p.scores = nullptr; p.map_out = nullptr; p.map_elem = 1; p.S = S; p.mode = mode; p.n_items = n_items;
  p.special = special_blocks < 0 ? 0 : (special_blocks > S ? S : special_blocks);
  p.causal = causal ? 1 : 0;
  double prev_hi = 0.0;
  for (int t = 0; t < PSA_MAX_LEVEL_ITEMS; ++t) {
    p.level[t] = 0; p.lo[t] = 0.f; p.hi[t] = 0.f;
  }
  for (int t = 0; t < n_items; ++t) {
    const int lv = item_level[t];
    PSA_REQUIRE(lv == 0 || lv == 1 || lv == 2 || lv == 4 || lv == 8, PSA_ERR_ARG, "psa_level_map_qwen: level %d not in {0,1,2,4,8}", lv);
    p.level[t] = lv;
    if (mode == PSA_MODE_THRESHOLDBOUND) {
      const double lower = item_lo[t] > prev_hi ? item_lo[t] : prev_hi;
      prev_hi = item_hi[t];
      p.lo[t] = (float)lower;
    } else {
      p.lo[t] = (float)item_lo[t];
    }
    p.hi[t] = (float)item_hi[t];
  }
  return PSA_OK;
}


// Host side: the kernel parameters of a level map with `Nk` columns (everything but the pointers).
static inline int level_map_fill_params(LevelMapParams& p, int Nk, int mode, int n_items, const int32_t* item_level,
                                        const double* item_hi, int align_div, int text_blocks, double min_full_attn_ratio) {
  PSA_REQUIRE(item_level && item_hi, PSA_ERR_ARG, "psa_level_map: mask_ratios must be provided");
  PSA_REQUIRE(mode == PSA_MODE_TOPK || mode == PSA_MODE_THRESHOLDBOUND, PSA_ERR_ARG,
              "Unknown mode: %d. Must be 'topk' or 'thresholdbound'", mode);
  PSA_REQUIRE(n_items >= 1 && n_items <= PSA_MAX_LEVEL_ITEMS, PSA_ERR_ARG, "psa_level_map: 1..%d items", PSA_MAX_LEVEL_ITEMS);
  PSA_REQUIRE(Nk > 0 && Nk <= 6144, PSA_ERR_UNSUPPORTED, "psa_level_map: Nk=%d out of range (Nk <= 6144)", Nk);
  PSA_REQUIRE(align_div >= 1 && text_blocks >= 0, PSA_ERR_ARG, "psa_level_map: bad align_div/text_blocks");
  p.scores = nullptr; p.map_out = nullptr; p.list_out = nullptr; p.map_elem = 4;
  p.Nk = Nk; p.mode = mode; p.n_items = n_items;
  p.text_blocks = text_blocks > Nk ? Nk : text_blocks;
  int m = (int)((double)Nk * min_full_attn_ratio) + 1;
  p.min_index = m < Nk ? m : Nk;
  int last_end = 0;
  for (int t = 0; t < PSA_MAX_LEVEL_ITEMS; ++t) {
    p.level[t] = 0; p.align[t] = 1; p.thr[t] = 0.f; p.fixed_s[t] = 0; p.fixed_e[t] = 0;
  }
  for (int t = 0; t < n_items; ++t) {
    const int lv = item_level[t];
    PSA_REQUIRE(lv == 0 || lv == 1 || lv == 2 || lv == 4 || lv == 8, PSA_ERR_ARG, "psa_level_map: level %d not in {0,1,2,4,8}", lv);
    p.level[t] = lv;
    const int al = (lv + align_div - 1) / align_div;  // ceil(level / (block_n / tile_n)); 0 for the skip level
    if (mode == PSA_MODE_THRESHOLDBOUND) {
      p.align[t] = al;
      p.thr[t] = (float)(item_hi[t] + 1e-6);
    } else {
      const int a = lv == 0 ? 1 : al;
      const int start = last_end;
      int end0 = (int)((double)Nk * item_hi[t]);
      end0 = end0 < Nk ? end0 : Nk;
      int end;
      const int len = end0 - start;
      if (a > 1 && len > 0) {
        const int rem = len % a;
        const int alen = rem ? len + (a - rem) : len;
        end = start + alen < Nk ? start + alen : Nk;
        if (end == Nk) end = start + ((end - start) / a) * a;
      } else {
        end = end0;
      }
      if (start < end) {
        p.fixed_s[t] = start; p.fixed_e[t] = end; last_end = end;
      } else {
        p.fixed_s[t] = start; p.fixed_e[t] = start;
      }
    }
  }
  p.n_cuts = 0;
  for (int t = 0; t < 2 * PSA_MAX_LEVEL_ITEMS; ++t) p.cut[t] = 0;
  for (int t = 0; t <= 2 * PSA_MAX_LEVEL_ITEMS; ++t) p.seg_level[t] = 0;
  if (mode == PSA_MODE_TOPK) {
    // the intervals are disjoint and in ascending order; ranks outside all of them are skipped (level 0)
    int at = 0, lvl = 0;  // level of the ranks from `at` on
    auto open = [&](int rank, int level) {
      if (level == lvl && rank > 0) return;
      if (rank > at) p.cut[p.n_cuts++] = rank;
      p.seg_level[p.n_cuts] = level;
      at = rank;
      lvl = level;
    };
    for (int t = 0; t < n_items; ++t)
      if (p.fixed_s[t] < p.fixed_e[t]) {
        open(p.fixed_s[t], p.level[t]);
        if (p.fixed_e[t] < Nk) open(p.fixed_e[t], 0);
      }
  }
  return PSA_OK;
}

// LDS scratch of level_map_row: of the selection where it serves the call (dense maps by quotas), else of the sort
static inline size_t level_map_lds_bytes(const LevelMapParams& p) {
  if (p.list_out == nullptr && level_map_selects(p.mode, p.n_cuts, p.Nk)) return SEL_LDS_BYTES;
  return sort_lds_bytes(p.Nk);
}
