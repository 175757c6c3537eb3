// DSA indexer KL loss in tiles of 64 query positions x 64 or 128 keys, bfloat16 / float16 query and key (gfx950).
//
// Same result as dsa_indexer_loss_mfma.hip, for callers that give a workspace: with the statistics of the
// softmaxes going through memory a row's keys are spread over workgroups, so that the causal triangle
// fills the CUs evenly, and no wavefront waits for another one's reductions:
//
//   dsa_loss_list_kernel    per row: membership bits of the index list, softmax statistics of the index scores (those
//                           by workgroups of the first pass where that is faster)
//   dsa_loss_tile_kernel<.., false>   per tile and head: sum of exp of the attention scores, per 64 keys
//   dsa_loss_merge_kernel   per (head, row): log2 of the softmax denominator over all its keys
//   dsa_loss_tile_kernel<.., true>    the scores again, p = mean over heads in registers, sum of p (log p - log q)
//   dsa_loss_sum_kernel     per row: the divergence summed over its 64-key chunks, in order
//
// In a tile a wavefront has 32 positions (columns of v_mfma_f32_32x32x16, one per lane) and 64 keys (rows);
// the heads' rows pass through LDS, fetched a step ahead as whole 16-byte pieces.  The masks
// (causal, membership, additive) sit in registers as addends of the one multiply-add that scales a score,
// and a lane reduces its own keys, so a head costs one lane exchange.
//
// Bound by the exponentials and the multiply-adds in front of them (two per pair and head; vector instructions fill 0.85 of
// the time in which all CUs have tiles).  Measured at 4096 positions, 8 heads of 64, lists of 1024: 80 us a call (lists 20: 84 MB
// read; passes 22 and 25, merge and sum 9), 84 with whole tiles only, 274 with a workgroup of 8 wavefronts per 16 positions
// (256 workgroups, the longest with twice the mean work, statistics in LDS per step).  Short sequences are bound by a
// workgroup's steps: 2 x 547 positions, 16 heads of 128 66 -> 34 us with split tiles, 943 x 8 x 128 44 -> 28.

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mfma_util.h"

namespace cm {
namespace {

constexpr int kThreads = 256;
constexpr int kQ = 64;                 // positions of a workgroup
constexpr int kChunk = 64;             // and keys
constexpr float kEps = 1e-10f;
constexpr size_t kPartBytes = 64u << 20;   // partial statistics of one slab of positions

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));       // rows of scores begin at any float

struct LossTiledParams {
  const unsigned short* q;   // [ASq, AB, AH, AD]
  const unsigned short* k;   // [Sk, AB, AH, AD]
  const float* index_scores; // [AB, ASq, Sk]
  const float* mask;         // [AB, ASq, Sk] or NULL
  const void* topk_idx;      // [AB, ASq, topk] or NULL
  float* loss;               // [AB, ASq]
  unsigned* bits;            // [AB, ASq, words] (lists only)
  float* index_norm;         // [AB, ASq]: log2 of the index softmax's denominator, max included
  float2* part;              // [chunks][AB * AH][slab rows]: max (base 2), sum
  float* norm;               // [AB * AH][slab rows]: log2 of the attention softmax's denominator, max included
  float* kl;                 // [chunks][AB][slab rows]
  void* range_event;         // recorded behind the kernel that reads the lists; or NULL
  int* range_flag;           // set to 1 when a list holds an index outside [0, Sk); or NULL
  unsigned char* outside;    // with range_flag: [rows, in whole workgroups of the list kernel], whether a row's list holds such an index
  int topk, index_dtype, words;
  int ASq, AB, AH, Sk;
  int slab0, slab_rows;      // positions of this slab
  int tiles;                 // of 64 positions x 128 keys of this slab and one batch
  int whole;                 // of all batches' tiles, those from here on are split
  int stats_rows;            // rows of index statistics that the first pass takes: all, or 0 (the list kernel takes them)
  int stats_groups;          // its workgroups for them
  long long first_tile;
  float scale2;              // softmax scale in base 2
};

template <bool F16>
__device__ __forceinline__ f32x16 product(const u32x4& a, const u32x4& b, const f32x16& c) {
  if (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// Rows from a base on, whose end the load unit checks: what lies behind it reads as zeros.
struct Rows {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ Rows(const char* base, unsigned bytes) : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, (int)bytes, 0x00020000)) {}
  __device__ u32x4 load(unsigned of_lane, int of_all) const { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)of_lane, of_all, 0)); }
};
__device__ __forceinline__ float exp2_(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float log2_(float x) { return __builtin_amdgcn_logf(x); }

// Softmax statistics of a row's index scores, by one wavefront; word_of(j): the membership bits from key j on.
template <int N, class Words>
__device__ __forceinline__ void index_statistics(const LossTiledParams& p, long long row, Words word_of) {
  const int lane = lane_id();
  const float* src = p.index_scores + (size_t)row * p.Sk;
  const float* add = p.mask ? p.mask + (size_t)row * p.Sk : nullptr;
  float m = -INFINITY, d = 0.0f;
  // N quads at a time, all requested before the first is looked at (NaN scores are skipped)
  for (int j0 = lane * 4; j0 < p.Sk; j0 += N * 256) {
    f32x4 v[N];
    unsigned word[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int j = j0 + n * 256;
      v[n] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      word[n] = 15u;
      if (j < p.Sk) {
        if (j + 3 < p.Sk) v[n] = *reinterpret_cast<const f32x4_any*>(src + j);
        else
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j + i < p.Sk) v[n][i] = src[j + i];
        word[n] = word_of(j);
      }
    }
    float top = m;
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (add && j0 + n * 256 + i < p.Sk) v[n][i] += add[j0 + n * 256 + i];
        if (!((word[n] >> i) & 1u)) v[n][i] = -INFINITY;
        if (v[n][i] > top) top = v[n][i];
      }
    if (top == -INFINITY) continue;
    d *= exp2_((m - top) * kLog2e);
    m = top;
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (v[n][i] > -INFINITY) d += exp2_((v[n][i] - top) * kLog2e);
  }
  const float top = wave_max(m);
  const float sum = wave_sum(m > -INFINITY ? d * exp2_((m - top) * kLog2e) : 0.0f);
  if (lane == 0) p.index_norm[row] = sum > 0.0f ? fmaf(top, kLog2e, log2_(sum)) : 0.0f;
}

// One wavefront per row: membership bits of the index list, and the statistics of the row where nothing else takes them.
// Many rows are bound by memory and by how many wavefronts wait for it: two quads on their way take 32 registers, eight take
// 108, half the wavefronts (5200 rows of 2600 scores with lists 25.6 -> 17.2 us, 7510 of 3755 34.1 -> 27.5; of 1000 rows, 7.6 -> 6.8).
__global__ __launch_bounds__(kThreads) void dsa_loss_list_kernel(const LossTiledParams p) {
  extern __shared__ unsigned lds_bits[];
  const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
  const long long row = (long long)blockIdx.x * 4 + wave;
  const bool live = row < (long long)p.AB * p.ASq;
  if (!p.topk_idx) {
    if (live) index_statistics<2>(p, row, [](int) { return 15u; });
    return;
  }
  unsigned* bits = lds_bits + wave * p.words;
  for (int w = lane; w < p.words; w += 64) bits[w] = 0u;
  __syncthreads();
  bool outside = false;
  if (live) {
#pragma unroll 4
    for (int t = lane; t < p.topk; t += 64) {
      const size_t at = (size_t)row * p.topk + t;
      const long long c = p.index_dtype == CPPMEGA_MI355_I64 ? static_cast<const long long*>(p.topk_idx)[at]
                                                             : (long long)static_cast<const int*>(p.topk_idx)[at];
      if (c >= 0 && c < p.Sk) atomicOr(&bits[(int)(c >> 5)], 1u << (c & 31));
      else outside = true;
    }
    if (outside && p.range_flag) *p.range_flag = 1;
  }
  const bool any = __ballot(outside) != 0ull;
  if (p.outside && lane == 0) p.outside[row] = any;
  __syncthreads();
  if (!live) return;
  for (int w = lane; w < p.words; w += 64) p.bits[(size_t)row * p.words + w] = bits[w];
  if (p.stats_rows == 0) index_statistics<2>(p, row, [&](int j) { return bits[j >> 5] >> (j & 31); });
}

// Tiles of 64 positions x 128 keys with a visible key in the first n blocks of positions (block i sees the keys of
// i / 2 + 1 tiles, at most all of them).
__host__ __device__ inline long long tiles_before(long long n, long long key_tiles) {
  const long long ramp = 2 * key_tiles, m = n < ramp ? n : ramp;
  return (m + 1) * (m + 1) / 4 + (n - m) * key_tiles;
}

// A tile of 64 positions; a wavefront has 32 positions (columns of v_mfma_f32_32x32x16, one per lane) and 64 keys (rows).
// Whole tiles of 128 keys: two halves of the positions by two of the keys, a head at a time.  Split ones of 64 keys: two
// halves of the positions by GROUPS groups of the heads, that many heads at a time.  Whole tiles pass 64 + 128 rows per head
// through LDS for 8192 pairs and set the masks up once for all heads; with less than a round of them what counts is a workgroup's
// time, which is its number of steps (1.6 us each, 4 us around them), and split ones have half as many.  GROUPS == 1: every
// tile is whole (three blocks of rows in LDS, not four: three workgroups on a CU for 128 channels); 2: the first p.whole
// are; 4: none is, where split tiles have a CU to themselves.
// GENERAL: an additive mask is given, or the softmax scale is not positive.  Otherwise the masks are 0 or -inf
// and enter the first pass as what its products start from (a select behind them where a row that does not count
// turned out not to be finite), and the second pass leaves keys that do not count out at its end.
// Workgroups of the first pass behind those of the tiles take the statistics of the index scores, a row to a wavefront (when, run()
// says).
// WIDE: 64 rows of scores are 2 GB and more, beyond the offsets of their descriptor, and are read by address (second pass; 130 positions of
// 8 heads of 64 over 2^23 keys 11.8 ms, 135 with a workgroup per 16 positions).
constexpr int kWideKeys = 1 << 23;
constexpr int resident(int AD, bool general) { return AD <= 64 && !general ? 4 : 2; }
template <bool F16, int AD, int GROUPS, bool SECOND, bool GENERAL, bool WIDE = false>
__global__ __launch_bounds__(GROUPS == 1 ? 256 : 128 * GROUPS, resident(AD, GENERAL)) void dsa_loss_tile_kernel(const LossTiledParams p) {
  constexpr bool WHOLE = GROUPS == 1;                     // whole tiles only
  constexpr int THREADS = WHOLE ? 256 : 128 * GROUPS, BLOCKS = WHOLE ? 3 : 2 * GROUPS;
  constexpr int PIECES = AD / 8;                          // 16-byte pieces of a row of one head
  constexpr int PITCH = PIECES + 1;                       // odd: 16 rows of a piece fall on 16 bank groups
  constexpr int LOADS = 64 * PIECES / THREADS;            // pieces of a thread of 64 rows of one head
  constexpr int STEPS = AD / 16;
  static_assert(LOADS * THREADS == 64 * PIECES, "whole pieces per thread");
  // 64 rows each: queries, keys of the first head, (split: queries,) keys of the second, ..; in the end the wavefronts' sums
  constexpr int BLOCK = 64 * PITCH, ROWS = BLOCKS * BLOCK, MEET = SECOND && !WHOLE ? 2 * GROUPS * 32 * 64 / 4 : 0;
  __shared__ u32x4 rows[ROWS > MEET ? ROWS : MEET];

  const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int id = (int)blockIdx.x;
  if (!SECOND && p.stats_rows) {
    // eights of workgroups, one per XCD: those of the tiles first
    const unsigned eight = (unsigned)id >> 3, tile_eights = (gridDim.x >> 3) - ((unsigned)(p.stats_groups + 7) >> 3);
    if (eight >= tile_eights) {
      const int row = ((int)(eight - tile_eights) * 8 + (id & 7)) * (THREADS / 64) + wave;
      if (row < p.stats_rows) {
        const unsigned* bits = p.bits + (size_t)row * p.words;
        index_statistics<8>(p, row, [&](int j) { return p.topk_idx ? bits[j >> 5] >> (j & 31) : 15u; });
      }
      return;
    }
  }
  // Tile of this workgroup: the causal triangles of the batches, one after the other.  Consecutive workgroups go round the
  // eight XCDs, and each XCD takes one run of tiles, whose query rows (and the keys) its L2 holds.
  const bool split = !WHOLE && (GROUPS > 2 || id >= p.whole);
  int within = id, count = p.whole;
  if (split) {
    within = id - p.whole;
    count = (p.tiles * p.AB - p.whole) * 2;
  }
  if (within >= count) return;
  const int share = count >> 3, rest = count & 7, xcd = within & 7;
  int at_tile = xcd * share + min(xcd, rest) + (within >> 3);
  const int key_half = split ? at_tile & 1 : 0;
  if (split) at_tile = p.whole + (at_tile >> 1);
  const int b = at_tile / p.tiles, key_tiles = (p.Sk + 127) / 128;
  const long long of_all = p.first_tile + (at_tile - b * p.tiles);
  int lo = p.slab0 / kQ, hi = (p.ASq + kQ - 1) / kQ;      // tiles_before(lo) <= of_all < tiles_before(hi)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (tiles_before(mid, key_tiles) <= of_all) lo = mid;
    else hi = mid;
  }
  const int q0 = lo * kQ, k0 = (int)(of_all - tiles_before(lo, key_tiles)) * 128 + key_half * 64;
  if (k0 > q0 + 63 || k0 >= p.Sk) return;                 // (the second half of a tile on the diagonal, or at the end)
  const int half = lane >> 5;
  const unsigned l32 = lane & 31;
  const int wq = (wave & 1) * 32, group = wave >> 1;
  const int kw = k0 + (split ? 0 : group * 64);          // the wavefront's first key
  const int my_q = q0 + wq + (int)l32;                         // the lane's position
  const bool live_q = my_q < p.ASq;
  const bool busy = kw <= q0 + wq + 31 && kw < p.Sk;      // the wavefront has a visible key
  const size_t row = (size_t)b * p.ASq + (live_q ? my_q : p.ASq - 1);
  const int steps = split ? (p.AH + GROUPS - 1) / GROUPS : p.AH;

  // rows of the tile, as far as there are any (the rest reads as zeros)
  const unsigned pos_bytes = (unsigned)p.AB * p.AH * AD * 2;
  const Rows q_rows(reinterpret_cast<const char*>(p.q) + (size_t)q0 * pos_bytes + (size_t)b * p.AH * AD * 2, (min(64, p.ASq - q0) - 1) * pos_bytes + p.AH * AD * 2);
  const Rows k_rows(reinterpret_cast<const char*>(p.k) + (size_t)k0 * pos_bytes + (size_t)b * p.AH * AD * 2, (min(128, p.Sk - k0) - 1) * pos_bytes + p.AH * AD * 2);
  unsigned src[LOADS];
  int dst[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int e = tid + i * THREADS, r = e / PIECES, c = e % PIECES;
    src[i] = (unsigned)r * pos_bytes + (unsigned)c * 16u;
    dst[i] = THREADS % PIECES ? r * PITCH + c : tid / PIECES * PITCH + tid % PIECES + i * (THREADS / PIECES * PITCH);
  }
  u32x4 piece[BLOCKS][LOADS];
  float norm_next = 0.0f;
  const int in_slab = q0 + wq - p.slab0;                  // a slab has whole tiles of positions
  const float* norm_src = SECOND ? p.norm + (size_t)b * p.AH * p.slab_rows + in_slab : nullptr;
  // (first pass of split tiles, 64 channels: the last 64 rows are requested behind the products, whose operands need the registers)
  constexpr bool LATE = !SECOND && GROUPS == 2 && AD == 64;
  auto fetch_rows = [&](auto split, int step, int from, int to) {     // rows of the blocks from .. to - 1
#pragma unroll
    for (int m = from; m < to; ++m) {
      const int h = split ? min(step * GROUPS + (m >> 1), p.AH - 1) : step;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        if (WHOLE) piece[m][i] = m ? k_rows.load(src[i] + (m == 2 ? 64u * pos_bytes : 0u), step * AD * 2) : q_rows.load(src[i], step * AD * 2);
        else if (m & 1) piece[m][i] = k_rows.load(src[i] + (split || m == 1 ? 0u : 64u * pos_bytes), h * AD * 2);
        else if (split || m == 0) piece[m][i] = q_rows.load(src[i], h * AD * 2);
      }
    }
  };
  auto fetch = [&](auto split, int step) {
    fetch_rows(split, step, 0, LATE ? BLOCKS - 1 : BLOCKS);
    if (SECOND) norm_next = (norm_src + (size_t)(split ? min(step * GROUPS + group, p.AH - 1) : step) * p.slab_rows)[l32];
  };
  // register v of a 32-key block: key 8 * (v / 4) + 4 * half + v % 4
  float add[2][16];
  unsigned counts[2];                                     // bit 8 * (v / 4) + v % 4: whether key v counts
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int key0 = kw + t * 32 + 4 * half;
    unsigned word = 0xffffffffu;
    if (p.topk_idx && (kw + t * 32) < p.Sk) word = p.bits[row * p.words + ((kw + t * 32) >> 5)] >> (4 * half);
    const int last = live_q ? min(my_q, p.Sk - 1) - key0 : -1;      // offsets up to here are visible
    counts[t] = last < 0 ? 0u : (last >= 31 ? word : word & ((2u << last) - 1u));
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int off = 8 * (v >> 2) + (v & 3);
      add[t][v] = (counts[t] >> off) & 1u ? 0.0f : -INFINITY;
      if (GENERAL && p.mask && add[t][v] == 0.0f) {
        const float x = p.mask[row * (size_t)p.Sk + key0 + off];
        add[t][v] = x > -INFINITY ? x * kLog2e : -INFINITY;
        if (!(x > -INFINITY)) counts[t] &= ~(1u << off);
      }
    }
  }

  float mean[2][16];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) mean[t][v] = 0.0f;

  // (split is a constant in the loop: as a run-time value its branches met again in front of the products, and all rows of the
  // step to come were waited for there)
  auto heads = [&](auto split) {
    const u32x4* const q_frag = rows + (split ? group : 0) * 2 * BLOCK + (wq + l32) * PITCH + half;
    const u32x4* const k_frag = rows + (1 + (WHOLE ? group : 2 * group)) * BLOCK + l32 * PITCH + half;
    fetch(split, 0);
    if (LATE) fetch_rows(split, 0, BLOCKS - 1, BLOCKS);
    for (int step = 0; step < steps; ++step) {
      __syncthreads();                                      // the previous heads' rows are read
#pragma unroll
      for (int m = 0; m < BLOCKS; ++m)
        if (WHOLE || m != 2 || split)
#pragma unroll
          for (int i = 0; i < LOADS; ++i) rows[m * BLOCK + dst[i]] = piece[m][i];
      const float norm = norm_next;
      fetch(split, min(step + 1, steps - 1));
      __syncthreads();
      const int h = split ? step * GROUPS + group : step;
      const bool takes = busy && h < p.AH;                  // (uniform)
      f32x16 s[2];
      auto products = [&](bool masked) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) s[t][v] = masked ? add[t][v] : 0.0f;
        if constexpr (AD > 64) {
          // Of the larger heads the operands are read a step ahead of their products: a wavefront is alone with one or two others
          // on its SIMD, and by itself the compiler waits for each (16 heads of 128, second pass, 272 tiles 36.5 -> 32.7 us, 1806
          // tiles 71.8 -> 67.6; up to 64 channels there are no registers for it: 28.7 -> 36.1).
          u32x4 qf[2], kf[2][2];
          auto read = [&](int k) {
            qf[k & 1] = q_frag[2 * k];
#pragma unroll
            for (int t = 0; t < 2; ++t) kf[k & 1][t] = k_frag[t * 32 * PITCH + 2 * k];
          };
          read(0);
          read(1);
#pragma unroll
          for (int k = 0; k < STEPS; ++k) {
#pragma unroll
            for (int t = 0; t < 2; ++t) s[t] = product<F16>(kf[k & 1][t], qf[k & 1], s[t]);
            if (k + 2 < STEPS) read(k + 2);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
#pragma unroll
          for (int k = 0; k < STEPS; ++k) {
            const u32x4 qf = q_frag[2 * k];
#pragma unroll
            for (int t = 0; t < 2; ++t) s[t] = product<F16>(k_frag[t * 32 * PITCH + 2 * k], qf, s[t]);
          }
        }
      };
      if (takes) products(!SECOND && !GENERAL);
      if (LATE) {
        __builtin_amdgcn_sched_barrier(0);
        fetch_rows(split, min(step + 1, steps - 1), BLOCKS - 1, BLOCKS);
      }
      if (!takes) continue;
      // (exponentials first, sums behind them: a sum right behind its exponential waits for it)
      if constexpr (SECOND) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int v = 0; v < 16; ++v) s[t][v] = exp2_(GENERAL ? fmaf(s[t][v], p.scale2, add[t][v]) - norm : fmaf(s[t][v], p.scale2, -norm));
#pragma unroll
          for (int v = 0; v < 16; ++v) mean[t][v] += s[t][v];
        }
      } else {
        float m, sum;
        auto statistics = [&]() {
          m = -INFINITY;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              if (GENERAL) s[t][v] = add[t][v] > -INFINITY ? fmaf(s[t][v], p.scale2, add[t][v]) : -INFINITY;
              m = fmaxf(m, s[t][v]);
            }
          m = fmaxf(m, xor32(m));
          if (!GENERAL) m *= p.scale2;
          // (the maximum comes off inside the multiply-add: a score rounded to float32 by itself is off by 2^-24 of its size,
          // which made the loss's error 1.7 times as large for scores of a spread of 1.4 in base 2 and 4 times for one of 8)
          const float at = m > -INFINITY ? m : 0.0f;
          float d[4];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int v = 0; v < 16; ++v) s[t][v] = exp2_(GENERAL ? s[t][v] - at : fmaf(s[t][v], p.scale2, -at));
#pragma unroll
            for (int v = 0; v < 16; ++v) d[v & 3] = t == 0 && v < 4 ? s[t][v] : d[v & 3] + s[t][v];
          }
          sum = (d[0] + d[1]) + (d[2] + d[3]);
          sum += xor32(sum);
        };
        statistics();
        // -inf + x is NaN where x is not finite: the row of a key that does not count holds such values, or a row that
        // counts does.  Only then the masks are applied behind the products.
        if (!GENERAL && __ballot(!(sum == sum)) != 0ull) {
          asm volatile("" ::: "memory");                    // (the operands are read again: kept from above, they would not fit)
          products(false);
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) s[t][v] = add[t][v] == 0.0f ? s[t][v] : -INFINITY;
          statistics();
          if (LATE) fetch_rows(split, min(step + 1, steps - 1), BLOCKS - 1, BLOCKS);   // (nor would these rows, kept over the above)
        }
        if (half == 0 && live_q) (p.part + ((size_t)(kw / kChunk) * p.AB * p.AH + (size_t)b * p.AH + h) * p.slab_rows + in_slab)[l32] = make_float2(m, sum);
      }
    }
  };
  if constexpr (WHOLE) heads(std::false_type{});
  else if (GROUPS > 2) heads(std::true_type{});
  else if (split) heads(std::true_type{});
  else heads(std::false_type{});
  if (!SECOND) return;

  const float inv_heads = 1.0f / (float)p.AH, index_norm = p.index_norm[row];
  // Keys 8 * g .. + 3 of block t: their index scores, all requested before the first is looked at (with a branch around each
  // quad and its loads the second pass took 1709 vector instructions a wavefront, half of them here, for 1365), ..
  const Rows s_rows(reinterpret_cast<const char*>(p.index_scores + ((size_t)b * p.ASq + q0) * p.Sk), (unsigned)min(64, p.ASq - q0) * (unsigned)p.Sk * 4u);
  const unsigned s_lane = ((unsigned)(my_q - q0) * (unsigned)p.Sk + (unsigned)(kw + 4 * half)) * 4u;
  auto scores_of = [&](int t, int g) {
    if constexpr (WIDE) {
      const int key = kw + t * 32 + 8 * g + 4 * half;
      f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (key + i < p.Sk) v[i] = p.index_scores[row * (size_t)p.Sk + key + i];
      return v;
    }
    return __builtin_bit_cast(f32x4, s_rows.load(s_lane + (t * 32 + 8 * g) * 4u, 0));
  };
  // .. and their divergence, the heads' probabilities adding up to `sums`.  Keys that do not count leave no trace: scores that
  // are NaN have q = 0 (the maximum of NaN and -inf is -inf).
  auto divergence = [&](int t, int g, const f32x4& scores, const float (&sums)[4]) {
    const unsigned of_block = t ? counts[1] : counts[0];
    float kl = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool ok = (of_block >> (8 * g + i)) & 1u;
      float shift = -index_norm;
      if (GENERAL && ok && p.mask) shift = fmaf(p.mask[row * (size_t)p.Sk + kw + t * 32 + 8 * g + 4 * half + i], kLog2e, shift);
      const float pj = sums[i] * inv_heads, qj = exp2_(fmaxf(fmaf(scores[i], kLog2e, shift), -INFINITY));
      const float with = fmaf(pj, log2_(pj + kEps) - log2_(qj + kEps), kl);
      kl = ok ? with : kl;
    }
    return kl;
  };
  float kl = 0.0f;
  if (split) {
    if constexpr (!WHOLE) {
      // the groups of heads meet in LDS, and each finishes its share of the 32 registers
      constexpr int MINE = 32 / GROUPS;
      const int t = group * MINE / 16, g0 = group * MINE % 16 / 4;
      f32x4 scores[MINE / 4];
#pragma unroll
      for (int g = 0; g < MINE / 4; ++g) scores[g] = scores_of(t, g0 + g);
      float* const meet = reinterpret_cast<float*>(rows) + lane;               // [wavefront][register][lane]
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) meet[((wave * 2 + t) * 16 + v) * 64] = mean[t][v];
      __syncthreads();
#pragma unroll
      for (int g = 0; g < MINE / 4; ++g) {
        float sums[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int of = 0; of < GROUPS; ++of)
#pragma unroll
          for (int i = 0; i < 4; ++i) sums[i] += meet[(((of * 2 + (wave & 1)) * 2 + t) * 16 + 4 * (g0 + g) + i) * 64];
        kl += divergence(t, g0 + g, scores[g], sums);
      }
      kl += xor32(kl);
      __syncthreads();
      float* const ends = reinterpret_cast<float*>(rows) + wq + l32;
      if (half == 0) ends[group * 64] = kl;
      __syncthreads();
      if (group) return;
#pragma unroll
      for (int of = 1; of < GROUPS; ++of) kl += ends[of * 64];
    }
  } else {
    if (!busy) return;
    f32x4 scores[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) scores[t][g] = scores_of(t, g);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float sums[4] = {mean[t][4 * g], mean[t][4 * g + 1], mean[t][4 * g + 2], mean[t][4 * g + 3]};
        kl += divergence(t, g, scores[t][g], sums);
      }
    kl += xor32(kl);
  }
  if (half == 0 && live_q) (p.kl + ((size_t)(kw / kChunk) * p.AB + b) * p.slab_rows + in_slab)[l32] = kl * kLn2;
}

// 64 columns by 4 groups of chunks, met in LDS in order
__global__ __launch_bounds__(kThreads) void dsa_loss_merge_kernel(const LossTiledParams p) {
  __shared__ float2 met[4][64];
  const int lane = lane_id(), group = (int)(threadIdx.x >> 6);
  const long long i = (long long)blockIdx.x * 64 + lane;
  const long long total = (long long)p.AB * p.AH * p.slab_rows;      // (whole multiples of 64)
  const int q = p.slab0 + (int)(i % p.slab_rows);
  const int chunks = q < p.ASq ? (min(q + 1, p.Sk) + kChunk - 1) / kChunk : 0;
  float m = -INFINITY, d = 0.0f;
  auto take = [&](const float2 x) {
    const float top = fmaxf(m, x.x), at = top > -INFINITY ? top : 0.0f;
    d = d * exp2_(m - at) + x.y * exp2_(x.x - at);
    m = top;
  };
#pragma unroll 4
  for (int c = group; c < chunks; c += 4) take(p.part[(size_t)c * total + i]);
  met[group][lane] = make_float2(m, d);
  __syncthreads();
  if (group || q >= p.ASq) return;
  m = -INFINITY;
  d = 0.0f;
  for (int g = 0; g < 4; ++g) take(met[g][lane]);
  p.norm[i] = d > 0.0f ? m + log2_(d) : 0.0f;
}

__global__ __launch_bounds__(kThreads) void dsa_loss_sum_kernel(const LossTiledParams p) {
  __shared__ float met[4][64];
  const int lane = lane_id(), group = (int)(threadIdx.x >> 6);
  const long long i = (long long)blockIdx.x * 64 + lane;
  const long long total = (long long)p.AB * p.slab_rows;
  const int q = p.slab0 + (int)(i % p.slab_rows);
  const int chunks = q < p.ASq ? (min(q + 1, p.Sk) + kChunk - 1) / kChunk : 0;
  // the caller is told of an index outside the range, and finds the losses as they were
  int outside = 0;
  if (p.outside) {
    const int words = (int)(((long long)p.AB * p.ASq + 3) / 4);
#pragma unroll 4
    for (int w = threadIdx.x; w < words; w += kThreads) outside |= reinterpret_cast<const int*>(p.outside)[w];
  }
  float kl = 0.0f;
#pragma unroll 4
  for (int c = group; c < chunks; c += 4) kl += p.kl[(size_t)c * total + i];
  met[group][lane] = kl;
  if (__syncthreads_or(outside)) return;
  if (!group && q < p.ASq) p.loss[(i / p.slab_rows) * p.ASq + q] = (met[0][lane] + met[1][lane]) + (met[2][lane] + met[3][lane]);
}

struct Layout { size_t bits, outside, index_norm, part, norm, kl, bytes; int words, chunks, slab_rows; };

Layout layout(const cppmega_mi355_dsa_loss_args_t& a) {
  Layout l;
  const size_t rows = (size_t)a.batch * a.seq_q, heads = (size_t)a.batch * a.heads;
  l.words = (a.seq_k + 31) / 32;
  l.chunks = (int)((std::min(a.seq_q, a.seq_k) + kChunk - 1) / kChunk);
  // the partial statistics grow with the square of the length: positions go in slabs
  const size_t per_row = heads * l.chunks * sizeof(float2);
  size_t slab = kPartBytes / per_row / kQ * kQ;
  slab = slab < kQ ? kQ : slab;
  const size_t all = ((size_t)a.seq_q + kQ - 1) / kQ * kQ;
  l.slab_rows = (int)(slab < all ? slab : all);
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t here = at; at += (bytes + 255) & ~(size_t)255; return here; };
  l.bits = take(a.topk_indices ? rows * l.words * 4 : 0);
  l.outside = take(a.topk_indices ? (rows + 3) / 4 * 4 : 0);
  l.index_norm = take(rows * 4);
  l.part = take(per_row * l.slab_rows);
  l.norm = take(heads * l.slab_rows * 4);
  l.kl = take((size_t)l.chunks * a.batch * l.slab_rows * 4);
  l.bytes = at;
  return l;
}

template <bool F16, int AD, int GROUPS>
void passes(LossTiledParams p, long long workgroups, bool general, hipStream_t stream) {
  constexpr int waves = GROUPS == 1 ? 4 : 2 * GROUPS;
  p.stats_groups = (p.stats_rows + waves - 1) / waves;
  const dim3 grid((unsigned)workgroups), block(64 * waves), merge(kThreads);
  const dim3 with_statistics((unsigned)(p.stats_groups ? (workgroups + 7) / 8 * 8 + (p.stats_groups + 7) / 8 * 8 : workgroups));
  const long long columns = (long long)p.AB * p.slab_rows / 64;
  if (general) hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, GROUPS, false, true>), with_statistics, block, 0, stream, p);
  else hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, GROUPS, false, false>), with_statistics, block, 0, stream, p);
  hipLaunchKernelGGL(dsa_loss_merge_kernel, dim3((unsigned)(columns * p.AH)), merge, 0, stream, p);
  if (p.Sk >= kWideKeys) {
    if (general) hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, GROUPS, true, true, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, GROUPS, true, false, true>), grid, block, 0, stream, p);
  } else if (general) hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, GROUPS, true, true>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, GROUPS, true, false>), grid, block, 0, stream, p);
  hipLaunchKernelGGL(dsa_loss_sum_kernel, dim3((unsigned)columns), merge, 0, stream, p);
}

template <bool F16, int AD>
int run(LossTiledParams p, hipStream_t stream) {
  const bool general = p.mask || !(p.scale2 > 0.0f);
  const int key_tiles = (p.Sk + 127) / 128;
  const long long round = 256 * resident(AD, general);
  // (the lists' bits come first: the caller may be waiting for what that kernel finds)
  const size_t rows = (size_t)p.AB * p.ASq;
  // Tiles that are taken whole, of `all` ones.  Heads of up to 64 channels: whole rounds, and a rest of up to 9/16 of one (with
  // lists, whose kernel takes the statistics of the index scores beside them, 7/16) is split (dense, whole / split, 8 heads of
  // 64: 121 tiles 31.6 / 25.2 us, 361 39.2 / 37.7, 552 49.5 / 48.0, 702 52.4 / 54.8, 900 60.2 / 64.8; 16 heads: 46.5 / 30.8, 54.7 / 50.9, 70.4 /
  // 69.9, 74.5 / 81.1, 89.8 / 98.3; lists: 361 tiles 49.6 / 47.8 and 64.7 / 60.9, 450 52.3 / 52.8 and 68.0 / 67.6, 544 56.3 / 58.7 and 77.2 / 79.7).
  // Larger heads, of which three workgroups of whole tiles fit on a CU and two of split ones: all or none (16 heads of 128: 225
  // tiles 62.7 / 55.2, 272 75.2 / 76.0, 441 81.2 / 95.7, 900 149.8 / 176.2).
  auto whole_of = [&](long long all) {
    if (AD > 64) return 2 * all > round ? all : 0;
    const long long rest = all % round;
    return 16 * rest <= (p.topk_idx ? 7 : 9) * round ? all - rest : all;
  };
  // The statistics of the index scores go behind the tiles, where they fill what the last round leaves idle and read memory beside
  // exponentials.  Dense, they need no launch of their own then (a kernel in front / behind the tiles: 3300 positions x 16 heads of 64
  // 74.8 / 69.6 us, 1800 x 2 x 16 of 128 77.2 / 71.9, 2400 x 8 of 128 49.9 / 45.6, 1800 x 8 of 64 29.9 / 26.7, 350 19.2 / 18.9; of
  // 58 shapes three are slower, by 1 to 2 %).  With lists, whose kernel is there anyway, it takes enough to do beside them: 16 heads of 64 (1250
  // positions 38.4 / 35.7 us, 1932 48.9 / 45.9, 3171 82.1 / 79.7, 4096 109.6 / 106.8; 22 lengths 1.03x in the mean, none more than 1.5 % slower;
  // 8 heads 0.95 .. 1.05x), or split tiles that leave room for them, which they do up to a fifth of a round (8 heads of 64: 180 tiles
  // 39.0 / 36.8 us, 242 40.0 / 41.4, 450 52.8 / 56.1).  A workgroup of the larger heads keeps a CU or half of one (16 heads of 128: 64 tiles
  // 38.8 / 35.1, 121 42.1 / 47.3, 225 56.3 / 67.2; 300 .. 4096 positions of 8 0.98x in the mean, of 16 1.01x).
  const long long of_all_rows = tiles_before((p.ASq + kQ - 1) / kQ, key_tiles) * p.AB;
  const bool room = whole_of(of_all_rows) == 0 && (AD > 64 ? of_all_rows <= 64 : 5 * of_all_rows <= round);
  const bool in_tiles = p.slab_rows >= p.ASq && (!p.topk_idx || room || (AD <= 64 && p.AH >= 16));
  p.stats_rows = in_tiles ? (int)rows : 0;
  if (p.topk_idx || !in_tiles)
    hipLaunchKernelGGL(dsa_loss_list_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(kThreads), p.topk_idx ? 16 * (size_t)p.words : 0, stream, p);
  CM_HIP_CHECK(hipGetLastError());
  if (p.range_event) CM_HIP_CHECK(hipEventRecord((hipEvent_t)p.range_event, stream));
  for (p.slab0 = 0; p.slab0 < p.ASq; p.slab0 += p.slab_rows) {
    const int end = std::min(p.slab0 + p.slab_rows, p.ASq);
    p.first_tile = tiles_before(p.slab0 / kQ, key_tiles);
    p.tiles = (int)(tiles_before((end + kQ - 1) / kQ, key_tiles) - p.first_tile);
    const long long all = (long long)p.tiles * p.AB;
    p.whole = (int)whole_of(all);
    const long long workgroups = p.whole + (all - p.whole) * 2;
    if (p.whole == all) {
      passes<F16, AD, 1>(p, workgroups, general, stream);
      continue;
    }
    if constexpr (AD == 64 || AD == 128) {
      if (workgroups <= 256 && p.AH > 2) {
        passes<F16, AD, 4>(p, workgroups, general, stream);
        continue;
      }
    }
    passes<F16, AD, 2>(p, workgroups, general, stream);
  }
  CM_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace

// 16-bit rows of whole 32-channel groups; a row's membership bits in a quarter of 64 KiB of LDS
bool dsa_indexer_loss_tiled_supports(const cppmega_mi355_dsa_loss_args_t& a) {
  if (a.in_dtype != CPPMEGA_MI355_BF16 && a.in_dtype != CPPMEGA_MI355_F16) return false;
  if (a.head_dim != 32 && a.head_dim != 64 && a.head_dim != 96 && a.head_dim != 128) return false;
  if ((size_t)a.batch * a.heads * a.head_dim * 2 * 128 >= (1ull << 32)) return false;         // a tile's rows within 32-bit offsets
  if (a.batch > 65535 || (size_t)a.seq_q * a.batch == 0 || a.heads == 0 || a.seq_k == 0) return false;
  return !a.topk_indices || a.seq_k <= 131072;
}

size_t dsa_indexer_loss_tiled_workspace_bytes(const cppmega_mi355_dsa_loss_args_t& a) { return layout(a).bytes; }

int dsa_indexer_loss_tiled_launch(const cppmega_mi355_dsa_loss_args_t& a, hipStream_t stream) {
  const Layout l = layout(a);
  char* ws = static_cast<char*>(a.workspace);
  LossTiledParams p;
  p.q = static_cast<const unsigned short*>(a.query); p.k = static_cast<const unsigned short*>(a.key);
  p.index_scores = a.index_scores; p.mask = a.index_mask; p.topk_idx = a.topk_indices; p.loss = a.loss;
  p.bits = reinterpret_cast<unsigned*>(ws + l.bits); p.index_norm = reinterpret_cast<float*>(ws + l.index_norm);
  p.part = reinterpret_cast<float2*>(ws + l.part); p.norm = reinterpret_cast<float*>(ws + l.norm);
  p.kl = reinterpret_cast<float*>(ws + l.kl);
  p.range_flag = a.range_flag;
  p.outside = a.range_flag && a.topk_indices ? reinterpret_cast<unsigned char*>(ws + l.outside) : nullptr;
  p.topk = a.topk; p.index_dtype = a.index_dtype; p.words = l.words;
  p.ASq = a.seq_q; p.AB = a.batch; p.AH = a.heads; p.Sk = a.seq_k;
  p.slab0 = 0; p.slab_rows = l.slab_rows;
  p.scale2 = a.softmax_scale * kLog2e;
  p.range_event = a.range_event;
  const bool f16 = a.in_dtype == CPPMEGA_MI355_F16;
  switch (a.head_dim) {
    case 32: return f16 ? run<true, 32>(p, stream) : run<false, 32>(p, stream);
    case 64: return f16 ? run<true, 64>(p, stream) : run<false, 64>(p, stream);
    case 96: return f16 ? run<true, 96>(p, stream) : run<false, 96>(p, stream);
    default: return f16 ? run<true, 128>(p, stream) : run<false, 128>(p, stream);
  }
}

}  // namespace cm
