// DSA indexer KL loss in tiles of 64 query positions x 128 keys, bfloat16 / float16 query and key (gfx950).
//
// Same result as dsa_indexer_loss_mfma.hip, for callers that give a workspace: with the statistics of the
// softmaxes going through memory a row's keys are spread over workgroups, so that the causal triangle
// fills the CUs evenly, and no wavefront waits for another one's reductions:
//
//   dsa_loss_list_kernel    per row: membership bits of the index list, softmax statistics of the index scores
//   dsa_loss_tile_kernel<.., false>   per tile and head: max and sum of exp of the attention scores, per 64 keys
//   dsa_loss_merge_kernel   per (head, row): log2 of the softmax denominator over all its keys
//   dsa_loss_tile_kernel<.., true>    the scores again, p = mean over heads in registers, sum of p (log p - log q)
//   dsa_loss_sum_kernel     per row: the divergence summed over its 64-key chunks, in order
//
// In a tile a wavefront has 32 positions (columns of v_mfma_f32_32x32x16, one per lane) and 64 keys (rows);
// the head's 64 + 128 rows pass through LDS, fetched one head ahead as whole 16-byte pieces.  The masks
// (causal, membership, additive) sit in registers as addends of the one multiply-add that scales a score,
// and a lane reduces its own keys, so a head costs one lane exchange.
//
// Bound by the exponentials and the multiply-adds in front of them (two per pair and head).  Measured at
// 4096 positions, 8 heads of 64, lists of 1024: 92 us a call (lists 16, passes 26 and 31, merge and sum 10),
// against 274 us with a workgroup of 8 wavefronts per 16 positions (256 workgroups, the longest with twice the
// mean work, statistics in LDS per step).

#include <algorithm>

#include "common.h"
#include "mfma_util.h"

namespace cm {
namespace {

constexpr int kThreads = 256;
constexpr int kQ = 64, kK = 128;       // positions and keys of a workgroup
constexpr int kChunk = 64;             // keys of a wavefront
constexpr float kEps = 1e-10f;
constexpr size_t kPartBytes = 64u << 20;   // partial statistics of one slab of positions

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

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
  int* range_flag;           // set to 1 when a list holds an index outside [0, Sk); or NULL
  unsigned char* outside;    // with range_flag: [rows, in whole workgroups of the list kernel], whether a row's list holds such an index
  int topk, index_dtype, words;
  int ASq, AB, AH, Sk;
  int slab0, slab_rows;      // positions of this slab
  float scale2;              // softmax scale in base 2
};

template <bool F16>
__device__ __forceinline__ f32x16 product(const u32x4& a, const u32x4& b, const f32x16& c) {
  if (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float exp2_(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float log2_(float x) { return __builtin_amdgcn_logf(x); }

// One wavefront per row.
__global__ __launch_bounds__(kThreads) void dsa_loss_list_kernel(const LossTiledParams p) {
  extern __shared__ unsigned lds_bits[];
  const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
  const long long row = (long long)blockIdx.x * 4 + wave;
  const bool live = row < (long long)p.AB * p.ASq;
  unsigned* bits = lds_bits + wave * p.words;
  const bool sparse = p.topk_idx != nullptr;
  if (sparse) {
    for (int w = lane; w < p.words; w += 64) bits[w] = 0u;
    __syncthreads();
    bool outside = false;
    if (live) {
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
    if (live)
      for (int w = lane; w < p.words; w += 64) p.bits[(size_t)row * p.words + w] = bits[w];
  }
  if (!live) return;
  const float* src = p.index_scores + (size_t)row * p.Sk;
  const float* add = p.mask ? p.mask + (size_t)row * p.Sk : nullptr;
  float m = -INFINITY, d = 0.0f;
  auto take = [&](const float (&v)[4], int n) {              // (NaN scores are skipped)
    float top = m;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n && v[i] > top) top = v[i];
    if (top == -INFINITY) return;
    d *= exp2_((m - top) * kLog2e);
    m = top;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n && v[i] > -INFINITY) d += exp2_((v[i] - top) * kLog2e);
  };
  if ((p.Sk & 3) == 0 && ((uintptr_t)p.index_scores & 15) == 0) {
#pragma unroll 4
    for (int j = lane * 4; j < p.Sk; j += 256) {
      const f32x4 s = *reinterpret_cast<const f32x4*>(src + j);
      float v[4] = {s[0], s[1], s[2], s[3]};
      if (add)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += add[j + i];
      if (sparse) {
        const unsigned w = bits[j >> 5] >> (j & 31);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (w >> i) & 1u ? v[i] : -INFINITY;
      }
      take(v, 4);
    }
  } else {
    for (int j = lane; j < p.Sk; j += 64) {
      float v[4] = {src[j] + (add ? add[j] : 0.0f), 0.0f, 0.0f, 0.0f};
      if (sparse && !((bits[j >> 5] >> (j & 31)) & 1u)) v[0] = -INFINITY;
      take(v, 1);
    }
  }
  const float top = wave_max(m);
  const float sum = wave_sum(m > -INFINITY ? d * exp2_((m - top) * kLog2e) : 0.0f);
  if (lane == 0) p.index_norm[row] = sum > 0.0f ? fmaf(top, kLog2e, log2_(sum)) : 0.0f;
}

// Tiles with a visible key in the first n blocks of positions (block i sees the keys of i / 2 + 1 tiles, at
// most all of them).
__host__ __device__ inline long long tiles_before(long long n, long long key_tiles) {
  const long long ramp = 2 * key_tiles, m = n < ramp ? n : ramp;
  return (m + 1) * (m + 1) / 4 + (n - m) * key_tiles;
}

// GENERAL: an additive mask is given, or the softmax scale is not positive.  Otherwise the masks are 0 or -inf
// and enter the first pass as what its products start from (a select behind them where a row that does not count
// turned out not to be finite), and the second pass leaves keys that do not count out at its end.
template <bool F16, int AD, bool SECOND, bool GENERAL>
__global__ __launch_bounds__(kThreads, AD <= 64 && !GENERAL ? 4 : 2) void dsa_loss_tile_kernel(const LossTiledParams p) {
  constexpr int PIECES = AD / 8;                          // 16-byte pieces of a row of one head
  constexpr int PITCH = PIECES + 1;                       // odd: 16 rows of a piece fall on 16 bank groups
  constexpr int LOADS = (kQ + kK) * PIECES / kThreads;
  constexpr int STEPS = AD / 16;
  static_assert(LOADS * kThreads == (kQ + kK) * PIECES, "whole pieces per thread");
  __shared__ u32x4 rows[(kQ + kK) * PITCH];               // 64 query rows, then 128 key rows

  // Tile of this workgroup.  The causal triangle is one row of workgroups; consecutive ones go round the
  // eight XCDs, and each XCD takes one run of tiles, whose query rows (and the keys) its L2 holds.
  const int share = (int)gridDim.x >> 3, rest = (int)gridDim.x & 7, xcd = (int)blockIdx.x & 7;
  const long long key_tiles = (p.Sk + kK - 1) / kK;
  const long long at_tile = tiles_before(p.slab0 / kQ, key_tiles) + xcd * share + min(xcd, rest) + ((int)blockIdx.x >> 3);
  int lo = p.slab0 / kQ, hi = (p.ASq + kQ - 1) / kQ;      // tiles_before(lo) <= at_tile < tiles_before(hi)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (tiles_before(mid, key_tiles) <= at_tile) lo = mid;
    else hi = mid;
  }
  const int q0 = lo * kQ, k0 = (int)(at_tile - tiles_before(lo, key_tiles)) * kK, b = (int)blockIdx.y;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, half = lane >> 5;
  const int wq = (wave & 1) * 32, wk = (wave >> 1) * kChunk;
  const int my_q = q0 + wq + l32, kw = k0 + wk;           // the lane's position, the wavefront's first key
  const bool live_q = my_q < p.ASq;
  const bool busy = kw <= q0 + wq + 31 && kw < p.Sk;      // the wavefront has a visible key
  const size_t row = (size_t)b * p.ASq + (live_q ? my_q : p.ASq - 1);

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

  const size_t pos_bytes = (size_t)p.AB * p.AH * AD * 2;
  const char* const q_base = reinterpret_cast<const char*>(p.q) + (size_t)q0 * pos_bytes + (size_t)b * p.AH * AD * 2;
  const char* const k_base = reinterpret_cast<const char*>(p.k) + (size_t)k0 * pos_bytes + (size_t)b * p.AH * AD * 2;
  unsigned src[LOADS];
  int dst[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int e = tid + i * kThreads, r = e / PIECES, c = e % PIECES;
    const int at = r < kQ ? min(r, p.ASq - 1 - q0) : min(r - kQ, p.Sk - 1 - k0);
    src[i] = (unsigned)at * (unsigned)pos_bytes + (unsigned)c * 16u;
    dst[i] = r * PITCH + c;
  }
  u32x4 piece[LOADS];
  float norm_next = 0.0f;
  const float* norm_src = SECOND ? p.norm + (size_t)b * p.AH * p.slab_rows + (live_q ? my_q - p.slab0 : 0) : nullptr;
  auto fetch = [&](int h) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {                      // (the first 64 rows are whole pieces of queries for every head size)
      const char* base = i < kQ * PIECES / kThreads ? q_base : k_base;
      piece[i] = *reinterpret_cast<const u32x4*>(base + (size_t)h * AD * 2 + src[i]);
    }
    if (SECOND) norm_next = norm_src[(size_t)h * p.slab_rows];
  };

  float mean[2][16];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) mean[t][v] = 0.0f;

  fetch(0);
  for (int h = 0; h < p.AH; ++h) {
    __syncthreads();                                      // the previous head's rows are read
#pragma unroll
    for (int i = 0; i < LOADS; ++i) rows[dst[i]] = piece[i];
    const float norm = norm_next;
    fetch(h + 1 < p.AH ? h + 1 : h);
    __syncthreads();
    if (!busy) continue;
    f32x16 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[t][v] = SECOND || GENERAL ? 0.0f : add[t][v];
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
      const u32x4 qf = rows[(wq + l32) * PITCH + 2 * k + half];
#pragma unroll
      for (int t = 0; t < 2; ++t) s[t] = product<F16>(rows[(kQ + wk + t * 32 + l32) * PITCH + 2 * k + half], qf, s[t]);
    }
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
        const float at = m > -INFINITY ? m : 0.0f;
        float d[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int v = 0; v < 16; ++v) s[t][v] = exp2_(GENERAL ? s[t][v] - at : fmaf(s[t][v], p.scale2, -at));
#pragma unroll
          for (int v = 0; v < 16; ++v) d[v & 3] += s[t][v];
        }
        sum = (d[0] + d[1]) + (d[2] + d[3]);
        sum += xor32(sum);
      };
      statistics();
      // -inf + x is NaN where x is not finite: the row of a key that does not count holds such values, or a row that
      // counts does.  Only then the masks are applied behind the products.
      if (!GENERAL && __ballot(!(sum == sum)) != 0ull) {
        asm volatile("" ::: "memory");                    // (the operands are read again: kept from above, they would not fit)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) s[t][v] = 0.0f;
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
          const u32x4 qf = rows[(wq + l32) * PITCH + 2 * k + half];
#pragma unroll
          for (int t = 0; t < 2; ++t) s[t] = product<F16>(rows[(kQ + wk + t * 32 + l32) * PITCH + 2 * k + half], qf, s[t]);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) s[t][v] = add[t][v] == 0.0f ? s[t][v] : -INFINITY;
        statistics();
      }
      if (half == 0 && my_q - p.slab0 < p.slab_rows && live_q)
        p.part[((size_t)(kw / kChunk) * p.AB * p.AH + (size_t)b * p.AH + h) * p.slab_rows + (my_q - p.slab0)] = make_float2(m, sum);
    }
  }
  if (!SECOND || !busy) return;

  const bool vec = (p.Sk & 3) == 0 && ((uintptr_t)p.index_scores & 15) == 0;
  const float inv_heads = 1.0f / (float)p.AH, index_norm = p.index_norm[row];
  const float* scores = p.index_scores + row * (size_t)p.Sk;
  float kl = 0.0f;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int key = kw + t * 32 + 8 * g + 4 * half;
      if (!live_q || key > my_q || key >= p.Sk) continue;
      float iv[4];
      if (vec) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(scores + key);
#pragma unroll
        for (int i = 0; i < 4; ++i) iv[i] = x[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) iv[i] = key + i < p.Sk ? scores[key + i] : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (key + i > my_q || key + i >= p.Sk) continue;    // masked keys carry p = 0 and q = 0
        const bool ok = (counts[t] >> (8 * g + i)) & 1u;
        const float pj = ok ? mean[t][4 * g + i] * inv_heads : 0.0f;
        const float v = !ok ? -INFINITY : (GENERAL ? fmaf(iv[i], kLog2e, add[t][4 * g + i]) : iv[i] * kLog2e);
        const float qj = v > -INFINITY ? exp2_(v - index_norm) : 0.0f;
        kl += pj * (log2_(pj + kEps) - log2_(qj + kEps));
      }
    }
  kl += xor32(kl);
  if (half == 0 && live_q && my_q - p.slab0 < p.slab_rows)
    p.kl[((size_t)(kw / kChunk) * p.AB + b) * p.slab_rows + (my_q - p.slab0)] = kl * kLn2;
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

template <bool F16, int AD>
int run(LossTiledParams p, hipStream_t stream) {
  for (p.slab0 = 0; p.slab0 < p.ASq; p.slab0 += p.slab_rows) {
    const int end = std::min(p.slab0 + p.slab_rows, p.ASq), key_tiles = (p.Sk + kK - 1) / kK;
    const dim3 grid((unsigned)(tiles_before((end + kQ - 1) / kQ, key_tiles) - tiles_before(p.slab0 / kQ, key_tiles)), (unsigned)p.AB), block(kThreads);
    const long long columns = (long long)p.AB * p.slab_rows / 64;
    const bool general = p.mask || !(p.scale2 > 0.0f);
    if (general) hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, false, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, false, false>), grid, block, 0, stream, p);
    hipLaunchKernelGGL(dsa_loss_merge_kernel, dim3((unsigned)(columns * p.AH)), block, 0, stream, p);
    if (general) hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, true, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((dsa_loss_tile_kernel<F16, AD, true, false>), grid, block, 0, stream, p);
    hipLaunchKernelGGL(dsa_loss_sum_kernel, dim3((unsigned)columns), block, 0, stream, p);
  }
  CM_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace

// 16-bit rows of whole 32-channel groups; a row's membership bits in a quarter of 64 KiB of LDS
bool dsa_indexer_loss_tiled_supports(const cppmega_mi355_dsa_loss_args_t& a) {
  if (a.in_dtype != CPPMEGA_MI355_BF16 && a.in_dtype != CPPMEGA_MI355_F16) return false;
  if (a.head_dim != 32 && a.head_dim != 64 && a.head_dim != 96 && a.head_dim != 128) return false;
  if ((size_t)a.batch * a.heads * a.head_dim * 2 * kK >= (1ull << 32)) return false;          // a tile's rows within 32-bit offsets
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
  const size_t rows = (size_t)a.batch * a.seq_q;
  hipLaunchKernelGGL(dsa_loss_list_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(kThreads), a.topk_indices ? 16 * (size_t)l.words : 0, stream, p);
  CM_HIP_CHECK(hipGetLastError());
  if (a.range_event) CM_HIP_CHECK(hipEventRecord((hipEvent_t)a.range_event, stream));
  const bool f16 = a.in_dtype == CPPMEGA_MI355_F16;
  switch (a.head_dim) {
    case 32: return f16 ? run<true, 32>(p, stream) : run<false, 32>(p, stream);
    case 64: return f16 ? run<true, 64>(p, stream) : run<false, 64>(p, stream);
    case 96: return f16 ? run<true, 96>(p, stream) : run<false, 96>(p, stream);
    default: return f16 ? run<true, 128>(p, stream) : run<false, 128>(p, stream);
  }
}

}  // namespace cm
