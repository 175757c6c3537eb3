// Sparse MLA backward in separate steps over a workspace: bfloat16 or float16 operands (gfx950).
//
// sparse_mla_bwd_mfma.hip adds every (selected row, channel) of every query to dkv with a float32 atomic
// at the L2, which takes one element per channel and clock: 151 M adds are 0.47 ms whatever else runs.
// With a workspace the adds happen in LDS instead, and the steps that do not need each other's registers run
// at their own occupancy:
//
//   lists    per (query, group): its valid keys in order, and where each band of keys begins;
//   steps    per band: the pieces of up to 16 keys that the queries have in it, one after the other (workgroups of the next kernel);
//   scores   per (query, 16 heads): S = Q . K^T and dP = dO . K^T with the scores of all keys in registers,
//            softmax statistics and delta across the workgroup, then P and dS = sm_scale P (dP - delta) as two
//            16-bit planes each (hi = round(x), lo = round(x - hi), a term is good to 2^-17), and q and d_out by
//            channel, both as dkv's matrix instructions take them: a load is 1 KB in a row;
//   dq       per (query, 16 heads, 144 channels): dQ^T = K^T . dS^T over 32-key tiles staged in LDS (rows of 576 = 512 + 64
//            channels: in the kernel of the scores up to 256 keys, and up to 512 where there are few queries);
//   dkv      per (band, 64 channels, share of the steps): dS^T . Q + P^T . dO of every step, added to a
//            float32 tile in LDS, written out once;
//   sum      over the shares, when there are several.
//
// Nothing is added in an order that varies: the same input gives the same bits.
//
// Measured at q [1, 1024, 16, 576], kv [1, 4096, 1, 576], top-k 256: 150 .. 155 us (561 us with the atomics; under the profiler lists 6,
// scores and dq 68, dkv 71 .. 87, sum 9).  dkv is bound by the vector cache (27 M accesses of 64 bytes: 4 KB of q and d_out and
// about 1 KB of planes for a step's 9 keys of 16) and ends with the CUs whose three bands are all full; scores and dq by the
// gather of 302 MB of key rows each.

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mfma_util.h"
#include "sparse_mla_bwd_util.h"

namespace cm {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
// At most: 210 rows of 64 floats (one for nobody) are 52.5 KB of LDS, three tiles to a CU; how many there are is chosen by make_plan.
constexpr int kBandKeys = 209;
constexpr int kAhead = 4;              // steps on their way in a wavefront of dkv
constexpr int kStepGroup = 2 * kAhead; // steps come in whole rounds of dkv's two wavefronts
constexpr int kAgain = 1 << 30;        // mark of a slot whose key occurs earlier in the same 16 slots
constexpr int kHeads = 16;             // heads of an item
constexpr int kRowBytes = 128;         // of planes per key
constexpr size_t kSlabBytes = 192u << 20;

struct SplitParams {
  const unsigned short* q;      // [B, S, H, D]
  const unsigned short* kv;     // [B, Skv, G, D]
  const unsigned short* d_out;  // [B, S, H, d_v]
  const void* indices;          // [B, S, G, topk]
  const float* sm_scale_dev;
  void* dq;                     // [B, S, H, D]
  float* dkv;                   // [B, Skv, G, D]
  int* keys;                    // [lists][stride] ascending, -1 behind the last
  int* starts;                  // [lists][bands + 2]: first slot of each band, the number of keys, whether one is marked kAgain
  int* step_starts;             // [lists][bands]: each band's first step among the list's
  unsigned char* rows;          // [lists][list_steps][16]: the row of a slot's key in its tile of dkv, band by band in whole steps
  int* band_steps;              // the number of steps so far, then [B * G * bands][first, number]
  i32x4* steps;                 // byte offset of planes, 64 times the step's place in rows (| keys | 32 if one may be marked), byte offsets of by_channel, keys
  char* planes;                 // [lists][chunks][hi, lo][dS heads 0-7, 8-15, P heads 0-7, 8-15][stride][8]
  unsigned short* by_channel;   // [lists][chunks][D / 64][channel % 4][q heads 0-7, 8-15, d_out heads 0-7, 8-15][16 channels][8]
  float* part;                  // [shares][B, Skv, G, D]
  int dq_dtype, index_dtype;
  int B, S, H, G, Skv, topk, D, d_v;
  int channels;                 // D in whole tiles of dkv
  int s0, ns;                   // queries of this slab: s0 .. s0 + ns of every sequence; list = (b * ns + s - s0) * G + g
  int chunks;                   // of 16 heads per group
  int stride;                   // key slots per list: topk in whole tiles, and two tiles to read past
  int bands, band_keys, shares;
  int list_steps;               // at most, of 16 slots of one band
  unsigned dead_step;           // 64 times the place in rows of a step of no keys
  int accumulate;               // add to dkv
  float sm_scale;
};

static_assert(kBandKeys < 256, "rows are bytes, and row band_keys is that of slots of no key");

// ---- lists -----------------------------------------------------------------------------------
// A bit per cache row says which are named; what stands below a key's bit is its rank.  A list that names a key twice is
// sorted by bands and then to each key's rank within its band.  (For every list the latter took 7.4 us at 1024 x 256 of 4096 keys,
// 11.8 at 600 x 250 of 852, whose bands hold 50 keys of a list; 5.6 and 5.2 here.)
__global__ __launch_bounds__(kThreads) void bwd_lists_kernel(const SplitParams p) {
  extern __shared__ int smem_lists[];
  const int words = (p.Skv + 31) / 32;
  int* begin = smem_lists;                             // [bands]: the band's first slot
  int* fill = begin + p.bands;                         // [bands]: behind its last
  int* step_of = fill + p.bands;                       // [bands]: its first step
  int* loose = step_of + p.bands;                      // [topk]
  int* sorted = loose + p.topk;                        // [topk]
  unsigned* bits = reinterpret_cast<unsigned*>(sorted + p.topk);       // [words]
  int* below = reinterpret_cast<int*>(bits + words);   // [words]: keys in the words before
  __shared__ int sums[kThreads / 64], again;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const size_t list = blockIdx.x;
  const unsigned bs = blockIdx.x / (unsigned)p.G;
  const int g = (int)(blockIdx.x - bs * (unsigned)p.G), b = (int)(bs / (unsigned)p.ns), s = (int)(bs - (unsigned)b * (unsigned)p.ns);
  const size_t src = (((size_t)b * p.S + p.s0 + s) * p.G + g) * (size_t)p.topk;
  if (list == 0 && tid == 0) p.band_steps[0] = 0;
  if (list == 0 && tid < 16) p.rows[p.dead_step / 4 + tid] = (unsigned char)p.band_keys;
  int key[8];                                          // topk <= 2048
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = tid + i * kThreads;
    if (i * kThreads >= p.topk) {                      // (uniform)
      key[i] = -1;
      continue;
    }
    long long v = -1;
    if (k < p.topk)
      v = p.index_dtype == CPPMEGA_MI355_I64 ? static_cast<const long long*>(p.indices)[src + k] : (long long)static_cast<const int*>(p.indices)[src + k];
    key[i] = v >= 0 && v < p.Skv ? (int)v : -1;
  }
  for (int w = tid; w < words; w += kThreads) bits[w] = 0u;
  for (int r = tid; r < p.bands; r += kThreads) fill[r] = 0;
  if (tid == 0) again = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (key[i] >= 0) {
      const unsigned bit = 1u << (key[i] & 31);
      if (atomicOr(bits + (key[i] >> 5), bit) & bit) again = 1;
    }
  __syncthreads();
  const bool twice = again != 0;                       // (uniform)
  int valid;
  if (!twice) {
    const int per = (words + kThreads - 1) / kThreads, w0 = min(tid * per, words), w1 = min(w0 + per, words);
    int mine = 0;
    for (int w = w0; w < w1; ++w) mine += __popc(bits[w]);
    const int upto = (int)wave_inclusive_sum_dpp((unsigned)mine);
    if (lane == 63) sums[wave] = upto;
    __syncthreads();
    int at = upto - mine;
    valid = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {
      if (w < wave) at += sums[w];
      valid += sums[w];
    }
    for (int w = w0; w < w1; ++w) {
      below[w] = at;
      at += __popc(bits[w]);
    }
    __syncthreads();
    auto rank = [&](int k) { return below[k >> 5] + __popc(bits[k >> 5] & ((1u << (k & 31)) - 1u)); };
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (key[i] >= 0) sorted[rank(key[i])] = key[i];
    for (int r = tid; r < p.bands; r += kThreads) {
      begin[r] = r * p.band_keys < p.Skv ? rank(r * p.band_keys) : valid;              // (bands behind the end are empty)
      fill[r] = (r + 1) * p.band_keys < p.Skv ? rank((r + 1) * p.band_keys) : valid;
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (key[i] >= 0) atomicAdd(fill + key[i] / p.band_keys, 1);
    __syncthreads();
    if (tid < 64) {                                    // exclusive prefix, 64 bands at a time
      int base = 0;
      for (int r0 = 0; r0 < p.bands; r0 += 64) {
        const int r = r0 + lane, n = r < p.bands ? fill[r] : 0, upto = (int)wave_inclusive_sum((unsigned)n);
        if (r < p.bands) begin[r] = fill[r] = base + upto - n;
        base += __shfl(upto, 63, 64);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (key[i] >= 0) loose[atomicAdd(fill + key[i] / p.band_keys, 1)] = key[i];
    __syncthreads();
    valid = fill[p.bands - 1];                         // (where its keys end now)
    for (int e = tid; e < valid; e += kThreads) {
      const int v = loose[e], first = begin[v / p.band_keys], last = fill[v / p.band_keys];
      int at = first;
      for (int o = first; o < last; ++o) at += loose[o] < v || (loose[o] == v && o < e);
      sorted[at] = v;
    }
    __syncthreads();
    if (tid == 0) again = 0;                           // (from here on: whether a step of 16 holds a key twice)
  }
  int* starts = p.starts + list * (p.bands + 2);
  if (tid < 64) {
    int base = 0;
    for (int r0 = 0; r0 < p.bands; r0 += 64) {
      const int r = r0 + lane, first = r < p.bands ? begin[r] : 0, steps = r < p.bands ? (fill[r] - first + 15) / 16 : 0;
      const int upto = (int)wave_inclusive_sum((unsigned)steps);
      if (r < p.bands) {
        starts[r] = first;
        step_of[r] = base + upto - steps;
        p.step_starts[list * p.bands + r] = base + upto - steps;
      }
      base += __shfl(upto, 63, 64);
    }
    if (lane == 0) starts[p.bands] = valid;
  }
  __syncthreads();
  // a key that its step of 16 (from the band's first slot on) holds already is marked, and has no row
  int* out = p.keys + list * (size_t)p.stride;
  unsigned char* rows = p.rows + list * (size_t)p.list_steps * 16;
  for (int k = tid; k < p.stride; k += kThreads) {
    int v = -1;
    if (k < valid) {
      v = sorted[k];
      const int of = v / p.band_keys, nth = k - begin[of], row = v - of * p.band_keys;
      const bool marked = twice && (nth & 15) != 0 && sorted[k - 1] == v;
      unsigned char* at = rows + step_of[of] * 16 + nth;
      *at = (unsigned char)(marked ? p.band_keys : row);
      if (k + 1 == fill[of])
        for (int e = nth + 1; e & 15; ++e) *++at = (unsigned char)p.band_keys;
      if (marked) {
        v |= kAgain;
        again = 1;
      }
    }
    out[k] = v;
  }
  __syncthreads();
  if (tid == 0) starts[p.bands + 1] = again;
}

// ---- steps -----------------------------------------------------------------------------------
// A band to a workgroup, the first workgroups of the kernel of the scores, which needs none of it: 4 to 6 us as a launch of its own.
template <int THREADS>
__device__ void steps_of_band(const SplitParams& p, int of) {
  __shared__ int sums[THREADS / 64], base_of;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int band = of % p.bands, bg = of / p.bands, b = bg / p.G, g = bg - b * p.G;
  const int per = (p.ns + THREADS - 1) / THREADS, s0 = min(tid * per, p.ns), s1 = min(s0 + per, p.ns);
  auto row = [&](int s) { return p.starts + (((size_t)b * p.ns + s) * p.G + g) * (p.bands + 2); };
  int mine = 0;
  for (int s = s0; s < s1; ++s) mine += (row(s)[band + 1] - row(s)[band] + 15) / 16 * p.chunks;
  const int upto = (int)wave_inclusive_sum((unsigned)mine);
  if (lane == 63) sums[wave] = upto;
  __syncthreads();
  int at = upto - mine, all = 0;
  for (int w = 0; w < THREADS / 64; ++w) {
    if (w < wave) at += sums[w];
    all += sums[w];
  }
  const int padded = (all + kStepGroup - 1) / kStepGroup * kStepGroup;            // with steps whose rows are all dead
  if (tid == 0) {
    base_of = atomicAdd(p.band_steps, padded);
    p.band_steps[2 + 2 * of] = base_of;
    p.band_steps[3 + 2 * of] = padded;
  }
  __syncthreads();
  i32x4* out = p.steps + base_of;
  for (int e = all + tid; e < padded; e += THREADS) out[e] = i32x4{0, (int)p.dead_step, 0, 0};
  for (int s = s0; s < s1; ++s) {
    const size_t list = ((size_t)b * p.ns + s) * p.G + g;
    const int* st = row(s);
    const int end = st[band + 1], marked = st[p.bands + 1];
    unsigned row = ((unsigned)list * p.list_steps + p.step_starts[list * p.bands + band]) * 64;
    for (int t = st[band]; t < end; t += 16, row += 64)
      for (int c = 0; c < p.chunks; ++c) {
        const unsigned item = (unsigned)(list * p.chunks + c);
        out[at++] = i32x4{(int)(item * (unsigned)p.stride * kRowBytes + t * 16), (int)(row | min(end - t, 16) | (marked ? 32 : 0)),
                          (int)(item * (unsigned)p.channels * 64), (int)(((unsigned)list * p.stride + t) * 4)};
      }
  }
}

// Where a 16-byte piece of a row of 64 channels stands in LDS: piece ^ fold_piece(row).  The sixteen rows that an operand read
// takes together, one piece or those of neighbouring quarter wavefronts, fall on all eight places.
__device__ __forceinline__ int fold_piece(int row) { return ((((row >> 3) ^ (row >> 2)) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 1) & 1); }

// the key of a slot, -1 for none
__device__ __forceinline__ int plain_key(int slot) { return slot < 0 ? -1 : slot & ~kAgain; }

// sum / maximum over the 16 lanes of a row
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ float row_max(float v) {
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

template <bool F16>
__device__ __forceinline__ uint2 pack4(const float (&v)[4]) {
  return F16 ? make_uint2(pack_f16(v[0], v[1]), pack_f16(v[2], v[3])) : make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
}
// hi and lo planes of 4 values
template <bool F16>
__device__ __forceinline__ void planes_of(const float (&v)[4], uint2& hi_plane, uint2& lo_plane) {
  float hi[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = v[i] * PlaneScale<F16>::up;
    lo[i] = hi[i] - (F16 ? (float)(_Float16)hi[i] : (float)(__bf16)hi[i]);
  }
  hi_plane = pack4<F16>(hi);
  lo_plane = pack4<F16>(lo);
}
template <bool F16>
__device__ __forceinline__ void put_planes(char* at, size_t to_lo, const float (&v)[4]) {
  uint2 hi, lo;
  planes_of<F16>(v, hi, lo);
  *reinterpret_cast<uint2*>(at) = hi;
  *reinterpret_cast<uint2*>(at + to_lo) = lo;
}

struct Item {
  int g, b, chunk, h0, nh;
  size_t list, bs;
};
// (32-bit divisions: there are fewer than 2^31 items, and the 64-bit ones are long scalar chains)
__device__ __forceinline__ Item item_of(const SplitParams& p, unsigned i) {
  Item it;
  const unsigned list = i / (unsigned)p.chunks, bs = list / (unsigned)p.G;
  it.chunk = (int)(i - list * (unsigned)p.chunks);
  it.list = list;
  it.g = (int)(list - bs * (unsigned)p.G);
  it.b = (int)(bs / (unsigned)p.ns);
  const int s = (int)(bs - (unsigned)it.b * (unsigned)p.ns);
  it.bs = (size_t)it.b * p.S + p.s0 + s;
  const int hg = p.H / p.G;
  it.h0 = it.g * hg + it.chunk * kHeads;
  it.nh = min(kHeads, hg - it.chunk * kHeads);
  return it;
}

// Softmax statistics of heads 4 * kg + v over all keys: the scores of T tiles of a wavefront become exp2(score - maximum).
struct Stats { float inv_sum[4], delta[4]; };
template <int W, int T>
__device__ __forceinline__ Stats row_stats(float* met, f32x4 (&s)[T], const f32x4 (&dp)[T], float (&m)[4], int wave, int l16, int kg, int tiles) {
  // over the row of 16 lanes, then over the wavefronts
#pragma unroll
  for (int v = 0; v < 4; ++v) m[v] = row_max(m[v]);
  if (l16 == 0)
#pragma unroll
    for (int v = 0; v < 4; ++v) met[(wave * 16 + 4 * kg + v) * 3] = m[v];
  __syncthreads();
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    m[v] = -INFINITY;
    for (int w = 0; w < W; ++w) m[v] = fmaxf(m[v], met[(w * 16 + 4 * kg + v) * 3]);
    m[v] = m[v] > -INFINITY ? m[v] : 0.0f;
  }
  float l[4] = {0.f, 0.f, 0.f, 0.f}, dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < T; ++i) {
    if (wave + i * W >= tiles) break;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      s[i][v] = exp2f(s[i][v] - m[v]);
      l[v] += s[i][v];
      dot[v] = fmaf(s[i][v], dp[i][v], dot[v]);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    l[v] = row_sum(l[v]);
    dot[v] = row_sum(dot[v]);
  }
  if (l16 == 0)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      met[(wave * 16 + 4 * kg + v) * 3 + 1] = l[v];
      met[(wave * 16 + 4 * kg + v) * 3 + 2] = dot[v];
    }
  __syncthreads();
  Stats r;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float sum = 0.0f, d = 0.0f;
    for (int w = 0; w < W; ++w) {
      sum += met[(w * 16 + 4 * kg + v) * 3 + 1];
      d += met[(w * 16 + 4 * kg + v) * 3 + 2];
    }
    r.inv_sum[v] = sum > 0.0f ? 1.0f / sum : 0.0f;
    r.delta[v] = d * r.inv_sum[v];
  }
  return r;
}

// q and d_out by channel: lane (channel l16 of a block, kg): 8 heads of q (kg 0, 1) or of d_out (kg 2, 3)
template <int W>
__device__ __forceinline__ void by_channel(const SplitParams& p, const Item& it, const unsigned short* Qs, const unsigned short* Os, int Dp, int Dvp, int wave, int l16, int kg) {
  const int tr_row = l16 >> 2, tr_col = (l16 & 3) * 4, D = Dp - 8, dv = Dvp - 8;
  unsigned short* bc = p.by_channel + (it.list * p.chunks + it.chunk) * (size_t)p.channels * 32 + (l16 & 3) * 512 + kg * 128 + (l16 >> 2) * 8;
  for (int cb = wave; cb < D / 16; cb += W) {
    const bool has_v = cb * 16 < dv, from_q = kg < 2 || !has_v;      // (every lane issues the transposing read)
    const unsigned short* src = from_q ? Qs + (8 * (kg & 1) + tr_row) * Dp + cb * 16 + tr_col : Os + (8 * (kg - 2) + tr_row) * Dvp + cb * 16 + tr_col;
    bf16x8 v = join(lds_tr16(src), lds_tr16(src + 4 * (from_q ? Dp : Dvp)));
    if (kg >= 2 && !has_v) v = zero8();
    *reinterpret_cast<bf16x8*>(bc + (size_t)(cb >> 2) * 2048 + (cb & 3) * 32) = v;
  }
}

// ---- scores ------------------------------------------------------------------------------------
// W wavefronts take the 16-key tiles in turn, up to T each.  A tile's rows come 32 channels at a time, four lanes
// to a row (a load of 64 rows' pieces is served a lane at a time: 53 us for the form that read its operands
// straight from memory), and go through 1 KB of LDS of the wavefront's own, so there is no barrier in the loop.
// A lane ends up with 4 heads of one key.
constexpr int kQueue = 6;                              // pieces of 32 channels on their way

template <bool F16, int W, int T>
__global__ __launch_bounds__(W * 64, 4) void bwd_scores_kernel(const SplitParams p) {
  const int step_groups = p.B * p.G * p.bands;
  if ((int)blockIdx.x < step_groups) {
    steps_of_band<W * 64>(p, (int)blockIdx.x);
    return;
  }
  extern __shared__ __align__(16) unsigned char smem[];
  const int D = p.D, dv = p.d_v, Dp = D + 8, Dvp = dv + 8;
  unsigned short* Qs = reinterpret_cast<unsigned short*>(smem);       // [16][Dp]
  unsigned short* Os = Qs + kHeads * Dp;                              // [16][Dvp]
  float* met = reinterpret_cast<float*>(Os + kHeads * Dvp);           // [W][16][3]
  unsigned short* pieces = reinterpret_cast<unsigned short*>(met + W * kHeads * 3);       // [W][16 keys][32]
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, kg = lane >> 4;
  const Item it = item_of(p, blockIdx.x - (unsigned)step_groups);
  const float sm_scale = p.sm_scale_dev ? *p.sm_scale_dev : p.sm_scale;
  const float scale2 = sm_scale * kLog2e;
  const int* keys = p.keys + it.list * (size_t)p.stride;
  const int valid = p.starts[it.list * (p.bands + 2) + p.bands], tiles = (valid + 15) / 16;

  for (int e = tid; e < kHeads * (D / 8); e += W * 64) {
    const int h = e / (D / 8), c = e - h * (D / 8);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (h < it.nh) v = *reinterpret_cast<const u32x4*>(p.q + (it.bs * p.H + it.h0 + h) * (size_t)D + c * 8);
    *reinterpret_cast<u32x4*>(Qs + h * Dp + c * 8) = v;
  }
  for (int e = tid; e < kHeads * (dv / 8); e += W * 64) {
    const int h = e / (dv / 8), c = e - h * (dv / 8);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (h < it.nh) v = *reinterpret_cast<const u32x4*>(p.d_out + (it.bs * p.H + it.h0 + h) * (size_t)dv + c * 8);
    *reinterpret_cast<u32x4*>(Os + h * Dvp + c * 8) = v;
  }
  __syncthreads();

  const unsigned short* qa = Qs + l16 * Dp + 8 * kg;
  const unsigned short* oa = Os + l16 * Dvp + 8 * kg;
  f32x4 s[T], dp[T];
  float m[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  const int ks = D / 32, vs = dv / 32, groups = (ks + kQueue - 1) / kQueue;
  const int row = lane >> 2, col = lane & 3;
  unsigned short* put = pieces + wave * 512 + row * 32 + ((col ^ (-(row >> 2) & 3)) << 3);
  const unsigned short* get = pieces + wave * 512 + l16 * 32 + ((kg ^ (-(l16 >> 2) & 3)) << 3);
  const unsigned short* kv = p.kv + ((size_t)it.b * p.Skv * p.G + it.g) * (size_t)D + col * 8;
  auto row_of = [&](int t) { return kv + (size_t)max(plain_key(keys[min(t, tiles - 1) * 16 + row]), 0) * p.G * (size_t)D; };
  const unsigned short *cur = kv, *next = kv;
  u32x4 queue[kQueue];
  auto request = [&](int i, const unsigned short* at, int c) { queue[i] = *reinterpret_cast<const u32x4*>(at + min(c, ks - 1) * 32); };
  if (wave < tiles) {
    cur = row_of(wave);
#pragma unroll
    for (int i = 0; i < kQueue; ++i) request(i, cur, i);
  }
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int t = wave + i * W;
    if (t >= tiles) break;                             // (uniform)
    const int key = plain_key(keys[t * 16 + l16]);
    next = row_of(t + W);
    f32x4 sa = {0.f, 0.f, 0.f, 0.f}, da = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < groups; ++c0) {
      const bool last = c0 + 1 == groups;
#pragma unroll
      for (int q = 0; q < kQueue; ++q) {
        const int c = c0 * kQueue + q;
        *reinterpret_cast<u32x4*>(put) = queue[q];
        request(q, last ? next : cur, last ? q : c + kQueue);
        if (c < ks) {
          const bf16x8 k = lds_b128(get);
          sa = mm<F16>(lds_b128(qa + c * 32), k, sa);
          if (c < vs) da = mm<F16>(lds_b128(oa + c * 32), k, da);
        }
      }
    }
    cur = next;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      s[i][v] = key >= 0 ? sa[v] * scale2 : -INFINITY;
      m[v] = fmaxf(m[v], s[i][v]);
    }
    // (the slots behind a list's last key were fetched from row 0, which may hold anything)
#pragma unroll
    for (int v = 0; v < 4; ++v) dp[i][v] = key >= 0 ? da[v] : 0.0f;
  }
  const Stats stat = row_stats<W, T>(met, s, dp, m, wave, l16, kg, tiles);
  char* out = p.planes + (it.list * p.chunks + it.chunk) * (size_t)p.stride * kRowBytes + (size_t)(kg >> 1) * p.stride * 16 + 8 * (kg & 1);
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int t = wave + i * W;
    if (t >= tiles) break;
    float pv[4], ds[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      pv[v] = s[i][v] * stat.inv_sum[v];
      ds[v] = pv[v] * (dp[i][v] - stat.delta[v]) * sm_scale;
    }
    char* at = out + (size_t)(t * 16 + l16) * 16;
    put_planes<F16>(at, (size_t)p.stride * 64, ds);
    put_planes<F16>(at + (size_t)p.stride * 32, (size_t)p.stride * 64, pv);
  }
  by_channel<W>(p, it, Qs, Os, Dp, Dvp, wave, l16, kg);
}

// ---- dq ------------------------------------------------------------------------------------------
// A workgroup is one wavefront with up to 144 channels of an item: the K tiles it stages in LDS are its own, so
// nothing waits at a barrier (73 us for workgroups of four that shared 32 whole rows).
constexpr int kStep = 32;                              // keys per tile
constexpr int kBlocks = 9;                             // 16-channel blocks per wavefront
constexpr int kPieces = kStep * kBlocks * 2 / 64;      // 16-byte pieces of a tile per lane
// Bytes to a row: the rows that one transposing read takes together stand in different banks.
__device__ __forceinline__ int k_row(int row) { return row * 320 + (row & 8) * 4; }
constexpr int kKtile = kStep * 320 + 32;

// acc[j][v]: channel 16 * j + 4 * kg + v of head l16, from channel 16 b0 on; `own` is LDS of the wavefront's
template <bool F16>
__device__ __forceinline__ void put_dq(const SplitParams& p, const Item& it, char* own, f32x4 (&acc)[kBlocks], int b0, int blocks, int D, int lane, int l16, int kg) {
#pragma unroll
  for (int j = 0; j < kBlocks; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[j][v] *= PlaneScale<F16>::down;
  const size_t base = (it.bs * p.H + it.h0) * (size_t)D + b0 * 16;
  if (p.dq_dtype == CPPMEGA_MI355_F32) {
    if (l16 >= it.nh) return;
#pragma unroll
    for (int j = 0; j < kBlocks; ++j)
      if (j < blocks) *reinterpret_cast<f32x4*>((float*)p.dq + base + (size_t)l16 * D + j * 16 + 4 * kg) = acc[j];
    return;
  }
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) {
    const float v[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
    *reinterpret_cast<uint2*>(own + l16 * 304 + j * 32 + kg * 8) = p.dq_dtype == CPPMEGA_MI355_F16 ? pack4<true>(v) : pack4<false>(v);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  for (int e = lane; e < it.nh * (kBlocks * 2); e += 64) {
    const int h = e / (kBlocks * 2), c = e - h * (kBlocks * 2);
    if (c < blocks * 2)
      *reinterpret_cast<u32x4*>((unsigned short*)p.dq + base + (size_t)h * D + c * 8) = *reinterpret_cast<const u32x4*>(own + h * 304 + c * 16);
  }
}

template <bool F16>
__global__ __launch_bounds__(64, 3) void bwd_dq_kernel(const SplitParams p) {
  __shared__ __align__(16) char Ks[kKtile];
  __shared__ __align__(16) unsigned short Ss[2 * kStep * kHeads];     // [hi, lo][32 keys][16 heads]
  const int D = p.D, nblk = D / 16, parts = (nblk + kBlocks - 1) / kBlocks;
  const int lane = (int)threadIdx.x, l16 = lane & 15, kg = lane >> 4;
  const int part = (int)(blockIdx.x % parts), b0 = part * kBlocks, blocks = min(kBlocks, nblk - b0);
  const Item it = item_of(p, blockIdx.x / parts);
  const int* keys = p.keys + it.list * (size_t)p.stride;
  const int valid = p.starts[it.list * (p.bands + 2) + p.bands], steps = (valid + kStep - 1) / kStep;
  const char* planes = p.planes + (it.list * p.chunks + it.chunk) * (size_t)p.stride * kRowBytes;
  const unsigned short* kv = p.kv + ((size_t)it.b * p.Skv * p.G + it.g) * (size_t)D + b0 * 16;

  int piece_row[kPieces], piece_col[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int e = lane + i * 64;
    piece_row[i] = e / (kBlocks * 2);
    piece_col[i] = e - piece_row[i] * (kBlocks * 2);
  }
  const int s_key = lane & 31, s_half = lane >> 5;
  u32x4 pre[kPieces], pre_s[2];
  const u32x4 zero = {0u, 0u, 0u, 0u};
  int tile_keys = 0;
  auto fetch_keys = [&](int step) { tile_keys = plain_key(keys[min(step * kStep + s_key, valid - 1)]); };
  auto fetch = [&](int step) {                         // of the keys in tile_keys
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int key = __shfl(tile_keys, piece_row[i], 64);
      pre[i] = *reinterpret_cast<const u32x4*>(kv + (size_t)key * p.G * (size_t)D + min(piece_col[i], blocks * 2 - 1) * 8);
    }
    const int pos = step * kStep + s_key;
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(planes + ((size_t)(pl * 4 + s_half) * p.stride + min(pos, valid - 1)) * 16);
      pre_s[pl] = pos < valid ? v : zero;
    }
  };
  f32x4 acc[kBlocks];
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
  if (steps) {
    fetch_keys(0);
    fetch(0);
    fetch_keys(1);
  }
  for (int step = 0; step < steps; ++step) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u32x4*>(Ks + k_row(piece_row[i]) + piece_col[i] * 16) = pre[i];
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) *reinterpret_cast<u32x4*>(Ss + (pl * kStep + s_key) * kHeads + s_half * 8) = pre_s[pl];
    __syncthreads();
    fetch(step + 1);                                   // (behind the last: its keys again)
    fetch_keys(step + 2);
    bf16x8 ds[2];
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) {
      const unsigned short* src = Ss + (pl * kStep + 8 * kg + tr_row) * kHeads + tr_col;
      ds[pl] = join(lds_tr16(src), lds_tr16(src + 4 * kHeads));
    }
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
      const unsigned short* src = reinterpret_cast<const unsigned short*>(Ks + k_row(8 * kg + tr_row)) + j * 16 + tr_col;
      const bf16x8 k = join(lds_tr16(src), lds_tr16(src + 4 * 160));
      acc[j] = mm<F16>(k, ds[0], acc[j]);
      acc[j] = mm<F16>(k, ds[1], acc[j]);
    }
    __syncthreads();
  }
  put_dq<F16>(p, it, Ks, acc, b0, blocks, D, lane, l16, kg);
}

// ---- scores and dq of 576 = 512 + 64 channels ---------------------------------------------------
// The two kernels above in one, for up to 64 W keys: a wavefront scores up to four tiles of 16 keys, two at a time; then it
// takes a quarter of the channels of all keys for dq, with dS of the other wavefronts out of LDS.  Eight
// wavefronts: four quarters of the channels by two halves of the tiles of 32 keys, added at the end.
// Measured against the two kernels: 79 queries x 8 heads x 160 of 7757 keys 25 -> 18 us, 512 x 64 x 256 of 2048 140 ->
// 120, 1024 x 16 x 256 of 4096 70 -> 67.  Bound by the key rows' way from the L2 (604 MB, of a cache of 4.7 MB that is a
// little more than an XCD's L2) and by the phases of a workgroup, two of which share a CU (77 KB of LDS each): 5 us until
// q, d_out and the first keys are there, 8 for the scores, 6 for statistics and planes, 9 for dq.  Neither half the
// loads in flight nor q and d_out in registers made a difference to the large shape.
constexpr int kD = 576, kDv = 512, kDp = kD + 8, kDvp = kDv + 8, kStage = 2, kStages = 5;       // pieces of 64 channels of a tile to a stage
constexpr int kFusedRows = kHeads * (kDp + kDvp) * 2;  // bytes of q and d_out, then of dS
template <int W> constexpr int kFusedLds = kFusedRows + W * (kHeads * 3 * 4 + kKtile) + W * 64 * 4;
static_assert(2 * kStage * 2048 <= kKtile && kStages * kStage >= kD / 64, "a stage of two tiles and 32 keys of dq share a wavefront's LDS");

template <bool F16, int W>
__global__ __launch_bounds__(W * 64, 2) void bwd_scores_dq_kernel(const SplitParams p) {
  const int step_groups = p.B * p.G * p.bands;
  if ((int)blockIdx.x < step_groups) {
    steps_of_band<W * 64>(p, (int)blockIdx.x);
    return;
  }
  constexpr int T = 4, kSlots = W * T * 16;
  static_assert(2 * kSlots * kHeads * 2 <= kFusedRows, "dS takes the place of q and d_out");
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned short* Qs = reinterpret_cast<unsigned short*>(smem);       // [16][kDp]
  unsigned short* Os = Qs + kHeads * kDp;                             // [16][kDvp]
  float* met = reinterpret_cast<float*>(smem + kFusedRows);           // [W][16][3]
  const int tid = (int)threadIdx.x, lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  char* own = reinterpret_cast<char*>(met + W * kHeads * 3) + wave * kKtile;
  int* list_keys = reinterpret_cast<int*>(reinterpret_cast<char*>(met + W * kHeads * 3) + W * kKtile);       // [64 W]
  const Item it = item_of(p, blockIdx.x - (unsigned)step_groups);
  const float sm_scale = p.sm_scale_dev ? *p.sm_scale_dev : p.sm_scale;
  const float scale2 = sm_scale * kLog2e;
  const int* keys = p.keys + it.list * (size_t)p.stride;
  const int valid = p.starts[it.list * (p.bands + 2) + p.bands], tiles = (valid + 15) / 16;
  const unsigned short* kv = p.kv + ((size_t)it.b * p.Skv * p.G + it.g) * (size_t)kD;
  const size_t key_step = (size_t)p.G * kD;

  // Two tiles at a time, two pieces of 64 channels of each per stage, eight lanes to a row (a load serves twice as much from
  // pieces of 128 bytes as of 64): two stages are on their way in registers while one passes through LDS to operand order.
  const int row = lane >> 3, col = lane & 7;
  unsigned short* put[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) put[r] = reinterpret_cast<unsigned short*>(own) + (row + 8 * r) * 64 + ((col ^ fold_piece(row + 8 * r)) << 3);
  const unsigned short* get[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) get[u] = reinterpret_cast<const unsigned short*>(own) + l16 * 64 + (((4 * u + kg) ^ fold_piece(l16)) << 3);
  int slot_row[T][2], slot_16[T];                      // (tiles behind the list's room are the last one again, and nobody looks)
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int* of_tile = keys + min(wave + i * W, p.stride / 16 - 1) * 16;
    slot_row[i][0] = of_tile[row];
    slot_row[i][1] = of_tile[row + 8];
    slot_16[i] = of_tile[l16];
  }
  const int slot_own = keys[min(tid, p.stride - 1)];
  // q and d_out, whole rows of neighbouring lanes
  constexpr int kQLoads = (kHeads * (kD / 8) + W * 64 - 1) / (W * 64), kOLoads = kHeads * (kDv / 8) / (W * 64);
  u32x4 staged[kQLoads + kOLoads];
#pragma unroll
  for (int i = 0; i < kQLoads + kOLoads; ++i) {
    const bool of_q = i < kQLoads;
    const int e = tid + (of_q ? i : i - kQLoads) * W * 64, per = (of_q ? kD : kDv) / 8, h = min(e / per, it.nh - 1), c = e - e / per * per;
    staged[i] = *reinterpret_cast<const u32x4*>((of_q ? p.q : p.d_out) + (it.bs * p.H + it.h0 + h) * (size_t)(of_q ? kD : kDv) + c * 8);
  }
  u32x4 queue[2][2][kStage][2];
  const unsigned short* rows_at[T][2];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int r = 0; r < 2; ++r) rows_at[i][r] = kv + (size_t)max(plain_key(slot_row[i][r]), 0) * key_step + col * 8;
  auto request = [&](auto pair_c, auto stage_c, bool one, bool two) {      // a stage of tiles 2 * pair and 2 * pair + 1
    constexpr int pair = decltype(pair_c)::value, stage = decltype(stage_c)::value;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (j ? two : one)                               // (uniform)
#pragma unroll
        for (int q = 0; q < kStage; ++q)
          if (stage * kStage + q < kD / 64)
#pragma unroll
            for (int r = 0; r < 2; ++r) queue[(pair * kStages + stage) & 1][j][q][r] = *reinterpret_cast<const u32x4*>(rows_at[2 * pair + j][r] + (stage * kStage + q) * 64);
  };
  using std::integral_constant;
  request(integral_constant<int, 0>{}, integral_constant<int, 0>{}, wave < tiles, wave + W < tiles);
  request(integral_constant<int, 0>{}, integral_constant<int, 1>{}, wave < tiles, wave + W < tiles);
#pragma unroll
  for (int i = 0; i < kQLoads + kOLoads; ++i) {
    const bool of_q = i < kQLoads;
    const int e = tid + (of_q ? i : i - kQLoads) * W * 64, per = (of_q ? kD : kDv) / 8, h = e / per, c = e - h * per;
    if (i == 0) list_keys[tid] = plain_key(slot_own);
    if (h < kHeads) *reinterpret_cast<u32x4*>((of_q ? Qs + h * kDp : Os + h * kDvp) + c * 8) = h < it.nh ? staged[i] : u32x4{0u, 0u, 0u, 0u};
  }
  __syncthreads();

  f32x4 s[T], dp[T];
  float m[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  const unsigned short *qa = Qs + l16 * kDp + 8 * kg, *oa = Os + l16 * kDvp + 8 * kg;
  auto score_pair = [&](auto pair_c, auto two_c) {     // two: both of its tiles have keys
    constexpr int pair = decltype(pair_c)::value;
    constexpr bool two = decltype(two_c)::value;
    f32x4 sa[2], da[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) sa[j] = da[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto stage_of = [&](auto stage_c) {
      constexpr int stage = decltype(stage_c)::value;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (j == 0 || two)
#pragma unroll
          for (int q = 0; q < kStage; ++q)
            if (stage * kStage + q < kD / 64)
#pragma unroll
              for (int r = 0; r < 2; ++r) *reinterpret_cast<u32x4*>(put[r] + (j * kStage + q) * 1024) = queue[(pair * kStages + stage) & 1][j][q][r];
      __builtin_amdgcn_wave_barrier();
      if constexpr (stage < kStages - 2) request(pair_c, integral_constant<int, stage + 2>{}, true, two);
      else if constexpr (pair == 0 && two) request(integral_constant<int, 1>{}, integral_constant<int, stage + 2 - kStages>{}, wave + 2 * W < tiles, wave + 3 * W < tiles);
      // (all of a stage's operands are read before its products, and whether there is a second tile is decided outside: with tests between
      // the products each waited for its own operands; with dq's loop below 41 shapes 1.013x, up to 1.04)
      constexpr int c0 = 2 * stage * kStage, steps = kD / 32 - c0 < 2 * kStage ? kD / 32 - c0 : 2 * kStage;       // of 32 channels
      bf16x8 a[steps], o[steps], k[2][steps];
#pragma unroll
      for (int qu = 0; qu < steps; ++qu) {
        a[qu] = lds_b128(qa + (c0 + qu) * 32);
        k[0][qu] = lds_b128(get[qu & 1] + (qu >> 1) * 1024);
        if (two) k[1][qu] = lds_b128(get[qu & 1] + (kStage + (qu >> 1)) * 1024);
        if (c0 + qu < kDv / 32) o[qu] = lds_b128(oa + (c0 + qu) * 32);
      }
#pragma unroll
      for (int qu = 0; qu < steps; ++qu)
#pragma unroll
        for (int j = 0; j < (two ? 2 : 1); ++j) {
          sa[j] = mm<F16>(a[qu], k[j][qu], sa[j]);
          if (c0 + qu < kDv / 32) da[j] = mm<F16>(o[qu], k[j][qu], da[j]);
        }
      __builtin_amdgcn_wave_barrier();
    };
    stage_of(integral_constant<int, 0>{});
    stage_of(integral_constant<int, 1>{});
    stage_of(integral_constant<int, 2>{});
    stage_of(integral_constant<int, 3>{});
    stage_of(integral_constant<int, 4>{});
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = 2 * pair + j;
      const bool counts = (j == 0 || two) && slot_16[i] >= 0;         // (the slots behind a list's last key were fetched from row 0, which may hold anything)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[i][v] = counts ? sa[j][v] * scale2 : -INFINITY;
        m[v] = fmaxf(m[v], s[i][v]);
        dp[i][v] = counts ? da[j][v] : 0.0f;
      }
    }
  };
  if (wave + W < tiles) score_pair(integral_constant<int, 0>{}, std::true_type{});
  else if (wave < tiles) score_pair(integral_constant<int, 0>{}, std::false_type{});
  if (wave + 3 * W < tiles) score_pair(integral_constant<int, 1>{}, std::true_type{});
  else if (wave + 2 * W < tiles) score_pair(integral_constant<int, 1>{}, std::false_type{});
  const Stats stat = row_stats<W, T>(met, s, dp, m, wave, l16, kg, tiles);
  by_channel<W>(p, it, Qs, Os, kDp, kDvp, wave, l16, kg);
  // P and dS: planes for dkv, and dS for the other wavefronts
  uint2 ds_hi[T], ds_lo[T];
  char* out = p.planes + (it.list * p.chunks + it.chunk) * (size_t)p.stride * kRowBytes + (size_t)(kg >> 1) * p.stride * 16 + 8 * (kg & 1);
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int t = wave + i * W;
    ds_hi[i] = ds_lo[i] = make_uint2(0u, 0u);
    if (t < tiles) {
      float pv[4], ds[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        pv[v] = s[i][v] * stat.inv_sum[v];
        ds[v] = pv[v] * (dp[i][v] - stat.delta[v]) * sm_scale;
      }
      char* at = out + (size_t)(t * 16 + l16) * 16;
      put_planes<F16>(at + (size_t)p.stride * 32, (size_t)p.stride * 64, pv);
      uint2 hi, lo;
      planes_of<F16>(ds, hi, lo);
      *reinterpret_cast<uint2*>(at) = hi;
      *reinterpret_cast<uint2*>(at + (size_t)p.stride * 64) = lo;
      if (t * 16 + l16 < valid) {
        ds_hi[i] = hi;
        ds_lo[i] = lo;
      }
    }
  }

  // ---- dq: quarter `part` of the channels, tiles of 32 keys first, first + W / 4, .. ----
  constexpr int kTurns = W / 4;
  const int part = wave & 3, first = wave >> 2, steps = (valid + kStep - 1) / kStep, b0 = part * kBlocks;
  const unsigned short* kv_part = kv + b0 * 16;
  int piece_row[kPieces], piece_col[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int e = lane + i * 64;
    piece_row[i] = e / (kBlocks * 2);
    piece_col[i] = e - piece_row[i] * (kBlocks * 2);
  }
  // two tiles are on their way
  u32x4 pre[2][kPieces];
  auto fetch = [&](int step, u32x4 (&to)[kPieces]) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int key = list_keys[min(step * kStep + piece_row[i], valid - 1)];
      to[i] = *reinterpret_cast<const u32x4*>(kv_part + (size_t)key * key_step + piece_col[i] * 8);
    }
  };
  if (first < steps) {
    fetch(first, pre[0]);
    fetch(first + kTurns, pre[1]);
  }
  __syncthreads();                                     // q and d_out are read
  unsigned short* Ss = Qs;                             // [hi, lo][kSlots][16 heads]
#pragma unroll
  for (int i = 0; i < T; ++i) {
    uint2* at = reinterpret_cast<uint2*>(Ss + ((wave + i * W) * 16 + l16) * kHeads + 4 * kg);
    at[0] = ds_hi[i];
    at[kSlots * kHeads / 4] = ds_lo[i];
  }
  __syncthreads();
  f32x4 acc[kBlocks];
#pragma unroll
  for (int j = 0; j < kBlocks; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tr_row = l16 >> 2, tr_col = (l16 & 3) * 4;
  auto turn = [&](int step, u32x4 (&of)[kPieces]) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u32x4*>(own + k_row(piece_row[i]) + piece_col[i] * 16) = of[i];
    __builtin_amdgcn_wave_barrier();
    fetch(step + 2 * kTurns, of);                      // (behind the last: its last key again)
    bf16x8 ds[2];
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) {
      const unsigned short* src = Ss + (pl * kSlots + step * kStep + 8 * kg + tr_row) * kHeads + tr_col;
      ds[pl] = join(lds_tr16(src), lds_tr16(src + 4 * kHeads));
    }
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
      const unsigned short* src = reinterpret_cast<const unsigned short*>(own + k_row(8 * kg + tr_row)) + j * 16 + tr_col;
      const bf16x8 k = join(lds_tr16(src), lds_tr16(src + 4 * 160));
      acc[j] = mm<F16>(k, ds[0], acc[j]);
      acc[j] = mm<F16>(k, ds[1], acc[j]);
    }
    __builtin_amdgcn_wave_barrier();
  };
  // (pairs without a branch between them: where a tile of pre[0] could follow another one the compiler would wait for all that is on
  // its way)
  const int turns = first < steps ? (steps - first + kTurns - 1) / kTurns : 0;
  for (int pair = 0; pair < turns / 2; ++pair) {
    turn(first + 2 * pair * kTurns, pre[0]);
    turn(first + (2 * pair + 1) * kTurns, pre[1]);
  }
  if (turns & 1) turn(first + (turns - 1) * kTurns, pre[0]);
  if (kTurns == 2) {
    if (first == 1)
#pragma unroll
      for (int j = 0; j < kBlocks; ++j) reinterpret_cast<f32x4*>(own)[j * 64 + lane] = acc[j];
    __syncthreads();
    if (first == 1) return;
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) acc[j] += reinterpret_cast<const f32x4*>(own + 4 * kKtile)[j * 64 + lane];
  }
  put_dq<F16>(p, it, own, acc, b0, kBlocks, kD, lane, l16, kg);
}

// ---- dkv -----------------------------------------------------------------------------------------
// A workgroup is two wavefronts and one band's tile, three workgroups to a CU.  The steps of a band are added one after
// the other (they may name the same key), with plain reads and writes: ds_add_f32 takes a lane at a time (1160 us for a
// form of this kernel that took 280 with a plain write in its place).  So the wavefronts take turns: while one reads its
// step's rows, adds and writes them, the other has its operands arrive and multiplies.  Four such workgroups of 150 keys took 82 us at the
// shape above and 135 with 64 heads (512 queries, 256 of 2048 keys), where one wavefront per band, four bands to a workgroup, took 86 and 160.
// 16 bytes per lane of whole rows meet in no bank.  Two wavefronts per band with 32 channels each read the planes twice (110 us); one per 16 channels
// of 600 keys, four times (315 us).
constexpr int kDkvThreads = 128;
// A base and 32-bit offsets: a scalar one per step, a lane's own for good.
struct Slab {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ explicit Slab(const void* base) : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000)) {}
  template <class T>
  __device__ T load(int of_lane, int of_all) const { return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rsrc, of_lane, of_all, 0)); }
  __device__ unsigned load32(int of_lane, int of_all) const { return __builtin_amdgcn_raw_buffer_load_b32(rsrc, of_lane, of_all, 0); }
};
template <bool F16>
__global__ __launch_bounds__(kDkvThreads, 2) void bwd_dkv_kernel(const SplitParams p) {
  extern __shared__ __align__(16) float tile[];        // [band_keys + 1][64], the last row for lanes of no key
  const int tid = (int)threadIdx.x, lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // consecutive tiles read the same planes and rows: an XCD (launches go round them) takes a run of tiles
  const int per_xcd = (int)gridDim.x / 8, work = (int)blockIdx.x % 8 * per_xcd + (int)blockIdx.x / 8;
  const int cols = (p.D + 63) / 64, band = work % p.bands, ch0 = work / p.bands % cols * 64;
  const int share = work / (p.bands * cols) % p.shares, bg = work / (p.bands * cols * p.shares);
  if (bg >= p.B * p.G) return;
  const int g = bg % p.G, b = bg / p.G;
  const int k0 = band * p.band_keys, rows = min(p.band_keys, p.Skv - k0);
  for (int e = tid; e < (p.band_keys + 1) * 16; e += kDkvThreads) reinterpret_cast<f32x4*>(tile)[e] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int* all = p.band_steps + 2 + 2 * (bg * p.bands + band);
  const int groups = __builtin_amdgcn_readfirstlane(all[1]) / kStepGroup;
  const int first = (int)((long long)groups * share / p.shares) * kStepGroup;
  const int n = ((int)((long long)groups * (share + 1) / p.shares) * kStepGroup - first) / 2;      // of this wavefront
  if (n > 0) {
    const i32x4* steps = p.steps + __builtin_amdgcn_readfirstlane(all[0]) + first + wave;          // every other one
    const unsigned plane_lane = ((unsigned)kg * p.stride + l16) * 16, lo_plane = (unsigned)p.stride * 64;
    const Slab planes(p.planes), rows_of(p.rows), by_channel(reinterpret_cast<const char*>(p.by_channel) + (size_t)ch0 * 64);
    char* const tile_lane = reinterpret_cast<char*>(tile) + l16 * 16;
    // a step's operands are on their way from its predecessor kAhead before it in the same registers: planes and rows
    // of q and d_out as soon as that one is multiplied, the places of its keys in the tile as soon as it is added
    bf16x8 hi[kAhead], lo[kAhead], qo[kAhead][4];
    unsigned slot[kAhead];                             // rows of keys 4 * kg + v in its bytes
    int row_word[kAhead], key_at[kAhead], row_word_of[kAhead], key_at_of[kAhead];
    i32x4 cur = steps[2 * min(lane, n - 1)], next = steps[2 * min(64 + lane, n - 1)];
    auto request = [&](int i, int at) {
      const int plane = __builtin_amdgcn_readlane(cur[0], at), operand = __builtin_amdgcn_readlane(cur[2], at);
      row_word[i] = __builtin_amdgcn_readlane(cur[1], at);
      key_at[i] = __builtin_amdgcn_readlane(cur[3], at);
      if (l16 < (row_word[i] & 31)) {                  // (the cache serves the lanes that ask)
        hi[i] = planes.load<bf16x8>(plane_lane, plane);
        lo[i] = planes.load<bf16x8>(plane_lane, plane + (int)lo_plane);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) qo[i][j] = by_channel.load<bf16x8>(lane * 16 + j * 1024, operand);
    };
    auto request_slots = [&](int i) {
      slot[i] = rows_of.load32(kg * 4, (int)((unsigned)row_word[i] >> 6) * 16);
      row_word_of[i] = row_word[i];
      key_at_of[i] = key_at[i];
    };
    f32x4 add[4];
    auto multiply = [&](int i, int ahead) {            // the step in registers i, which then take the step `ahead`
#pragma unroll
      for (int j = 0; j < 4; ++j) add[j] = mm<F16>(hi[i], qo[i][j], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int j = 0; j < 4; ++j) add[j] = mm<F16>(lo[i], qo[i][j], add[j]);
      if ((ahead & 63) == 0) {
        cur = next;
        next = steps[2 * min(ahead + 64 + lane, n - 1)];
      }
      request(i, ahead & 63);
    };
    auto add_up = [&](int i) {                         // keys 4 * kg + v, channels 4 * l16 + j
      f32x4 was[4], *at[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        at[v] = reinterpret_cast<f32x4*>(tile_lane + (slot[i] >> 8 * v & 0xff) * 256);
        was[v] = *at[v];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) *at[v] = was[v] + f32x4{add[0][v], add[1][v], add[2][v], add[3][v]};
      if (row_word_of[i] & 32) {                       // (a list that names a key twice)
        // the lanes of one kg at a time: the others may hold the same key, and the row each has added to is written
        // before the next one reads it (to a single thread the four rounds are one, hence the fences)
        auto turn = [] {
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
        };
        turn();
        const int* keys = p.keys + key_at_of[i] / 4 + kg * 4;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int slot_of = keys[v], row = (slot_of & ~kAgain) - k0;
          const bool again = slot_of >= 0 && (slot_of & kAgain) && row >= 0 && row < p.band_keys;   // (not of a band behind)
#pragma unroll 1
          for (int k = 0; k < 4; ++k) {
            if (again && kg == k) {
              f32x4* once_more = reinterpret_cast<f32x4*>(tile + row * 64) + l16;
              *once_more += f32x4{add[0][v], add[1][v], add[2][v], add[3][v]};
            }
            turn();
          }
        }
      }
      request_slots(i);
    };
    // what was added is in LDS before the other wavefront reads it; loads of global memory stay on their way
    auto pass_on = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      request(i, i);
      request_slots(i);
    }
    pass_on();                                         // the tile is cleared
    multiply(0, kAhead);
    if (wave) pass_on();                               // half a turn behind
    for (int step = 0; step < n; step += kAhead) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        add_up(i);
        pass_on();
        multiply((i + 1) % kAhead, step + i + 1 + kAhead);             // (behind the last step: one nobody adds)
        pass_on();
      }
    }
    if (!wave) pass_on();
  }
  __syncthreads();
  const bool whole = p.shares > 1;
  float* out = (whole ? p.part + (size_t)share * p.B * p.Skv * p.G * p.D : p.dkv) + ((size_t)b * p.Skv + k0) * p.G * (size_t)p.D + (size_t)g * p.D + ch0;
  const int quads = min(64, p.D - ch0) / 4;
  for (int e = tid; e < rows * 16; e += kDkvThreads) {
    const int row = e >> 4, c4 = e & 15;
    if (c4 >= quads) continue;
    f32x4 v = *reinterpret_cast<const f32x4*>(tile + row * 64 + c4 * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= PlaneScale<F16>::down;
    f32x4* dst = reinterpret_cast<f32x4*>(out + (size_t)row * p.G * p.D + c4 * 4);
    if (!whole && p.accumulate) v += *dst;
    *dst = v;
  }
}

__global__ __launch_bounds__(kThreads) void bwd_sum_kernel(const SplitParams p) {
  const size_t n = (size_t)p.B * p.Skv * p.G * p.D / 4, i = (size_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  f32x4* dst = reinterpret_cast<f32x4*>(p.dkv) + i;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (p.accumulate) v = *dst;
  for (int z = 0; z < p.shares; ++z) v += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.part) + (size_t)z * n + i);
  *dst = v;
}

struct Plan {
  int chunks, stride, bands, band_keys, shares, ns;
  size_t keys, starts, step_starts, rows, band_steps, steps, list_steps, planes, by_channel, part, slab_bytes, bytes;
};

// A CU holds three tiles of dkv: as many shares of the steps as bring the tiles to three times the number of CUs, of eight at least.
int shares_of(long long tiles, long long items, int topk, int bands) {
  return (int)std::max<long long>(1, std::min<long long>(768 / tiles, items * (topk / (bands * 16) + 1) / 8));
}

// Bands of a sequence's keys: the number with the least modelled time of what depends on it.  A list of n keys in a band is
// n / 16 + 1/2 steps in the mean, 0.266 us each, which the busiest of the 768 places of a tile takes one after the other (with 22
// bands of 9 columns three shares leave 174 places empty, with 21 four leave 12); the shares' sums cross memory twice; a band
// more costs the lists and steps 0.3 us.  Measured on 108 shapes (8 .. 64 heads, 64 .. 1024 queries, 64 .. 512 of 512 .. 8192 keys),
// up to nine numbers of bands each, whole calls: 0.4 % from the best of them in the mean, 1.8 % at most, and 4.4 % faster than bands
// of 204 keys whatever the shape (1000 queries x 32 heads x 400 of 5000 keys, 25 / 28 bands 442 / 420 us; 394 x 64 x 183 of 4302 22 / 21
// 231 / 208; 500 x 64 x 500 of 700 4 / 6 500 / 476; 1024 x 16 x 256 of 4096 21 / 22 157 / 171).  Four tiles of 150 keys on a CU keep more of
// the planes in flight than an XCD's L2 holds (900 x 64 x 500 of 8000 943 / 1080).
int choose_bands(const cppmega_mi355_sparse_mla_bwd_args_t& a) {
  const long long columns = (long long)(a.d_qk + 63) / 64 * a.batch * a.kv_groups, items = (long long)a.seq_q * ((a.heads / a.kv_groups + kHeads - 1) / kHeads);
  const int least = (a.seq_kv + kBandKeys - 1) / kBandKeys, most = std::min((a.seq_kv + 99) / 100, least + 48);
  const double sum_us = (double)a.batch * a.seq_kv * a.kv_groups * a.d_qk * 8 / 3.5e6;
  int best = least;
  double best_us = 0.0;
  for (int bands = least; bands <= most; ++bands) {
    const int shares = shares_of(bands * columns, items, a.topk, bands);
    const double n = (double)a.topk / bands, steps = items * std::min(n, n / 16 + 0.5) / shares;
    const double us = 0.266 * (double)((bands * columns * shares + 767) / 768) * steps + (shares > 1 ? shares * sum_us : 0.0) + 0.3 * bands;
    if (bands == least || us < best_us) {
      best = bands;
      best_us = us;
    }
  }
  return best;
}

Plan make_plan(const cppmega_mi355_sparse_mla_bwd_args_t& a) {
  Plan l;
  l.chunks = (a.heads / a.kv_groups + kHeads - 1) / kHeads;
  l.stride = (a.topk + 15) / 16 * 16 + 32;
  l.bands = choose_bands(a);
  l.band_keys = (a.seq_kv + l.bands - 1) / l.bands;
  const size_t lists = (size_t)a.batch * a.kv_groups, bands = (size_t)l.bands;               // lists per query position
  l.list_steps = a.topk / 16 + std::min<size_t>((size_t)a.topk, bands) + 1;
  const size_t per_s = lists * (l.stride * 4 + (2 * bands + 2) * 4 + l.list_steps * (16 + 16 * l.chunks) + l.chunks * ((size_t)l.stride * kRowBytes + (size_t)(a.d_qk + 63) / 64 * 4096));
  l.ns = (int)std::min<size_t>((size_t)a.seq_q, std::max<size_t>(kSlabBytes / per_s, 1));
  l.shares = shares_of((long long)l.bands * ((a.d_qk + 63) / 64) * lists, (long long)l.ns * l.chunks, a.topk, l.bands);
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t here = at; at += (bytes + 255) & ~(size_t)255; return here; };
  l.keys = take(lists * l.ns * l.stride * 4);
  l.starts = take(lists * l.ns * (bands + 2) * 4);
  l.band_steps = take((2 + lists * bands * 2) * 4);
  l.step_starts = take(lists * l.ns * bands * 4);
  l.rows = take((lists * l.ns * l.list_steps + 1) * 16);
  l.steps = take((lists * l.ns * l.list_steps * l.chunks + lists * bands * kStepGroup) * 16);
  l.planes = take(lists * l.ns * l.chunks * l.stride * kRowBytes);
  l.by_channel = take(lists * l.ns * l.chunks * ((a.d_qk + 63) / 64) * 4096);
  l.slab_bytes = at;
  l.part = take(l.shares > 1 ? (size_t)l.shares * a.batch * a.seq_kv * a.kv_groups * a.d_qk * 4 : 0);
  l.bytes = at;
  return l;
}

template <bool F16>
int run(SplitParams p, const Plan& l, bool clear, hipStream_t stream) {
  auto scores_lds = [&](int waves) { return (size_t)2 * kHeads * (p.D + 8 + p.d_v + 8) + waves * (kHeads * 3 * 4 + 1024); };
  const size_t dkv_lds = (size_t)(p.band_keys + 1) * 64 * 4;
  const int dq_parts = (p.D / 16 + kBlocks - 1) / kBlocks;
  // (all but the kernels of scores and dq together stay within the 64 KB that need no asking)
  const bool rows_of_576 = p.D == kD && p.d_v == kDv && p.topk <= 512;
  if (rows_of_576) {
    if (p.topk <= 256) CM_HIP_CHECK(hipFuncSetAttribute((const void*)bwd_scores_dq_kernel<F16, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, kFusedLds<4>));
    else CM_HIP_CHECK(hipFuncSetAttribute((const void*)bwd_scores_dq_kernel<F16, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, kFusedLds<8>));
  }
  for (p.s0 = 0; p.s0 < p.S; p.s0 += l.ns) {
    p.ns = std::min(l.ns, p.S - p.s0);
    p.shares = l.shares;
    p.accumulate = p.s0 > 0 || !clear;
    const size_t lists = (size_t)p.B * p.ns * p.G, items = lists * p.chunks;
    hipLaunchKernelGGL(bwd_lists_kernel, dim3((unsigned)lists), dim3(kThreads), (size_t)(3 * p.bands + 2 * p.topk + 2 * ((p.Skv + 31) / 32)) * 4, stream, p);
    const dim3 of_items((unsigned)(items + (size_t)p.B * p.G * p.bands));        // (and the bands' steps in front)
    // Of eight wavefronts with up to 512 keys a CU holds one workgroup: one kernel while that is one round, else two (rows of 3000 keys, one kernel
    // / two: 220 items x 350 27.5 / 36.5 us, 250 x 500 33.4 / 45.4, 376 x 438 55.9 / 53.7, 440 x 300 48.2 / 46.4, 2000 x 350 of 4000 215 / 194).
    const bool fused = rows_of_576 && (p.topk <= 256 || items <= 256);
    if (fused) {
      if (p.topk <= 256) hipLaunchKernelGGL((bwd_scores_dq_kernel<F16, 4>), of_items, dim3(256), kFusedLds<4>, stream, p);
      else hipLaunchKernelGGL((bwd_scores_dq_kernel<F16, 8>), of_items, dim3(512), kFusedLds<8>, stream, p);
    } else if (p.topk <= 16 * 4 * 4) hipLaunchKernelGGL((bwd_scores_kernel<F16, 4, 4>), of_items, dim3(256), scores_lds(4), stream, p);
    else if (p.topk <= 16 * 8 * 4) hipLaunchKernelGGL((bwd_scores_kernel<F16, 8, 4>), of_items, dim3(512), scores_lds(8), stream, p);
    else hipLaunchKernelGGL((bwd_scores_kernel<F16, 16, 8>), of_items, dim3(1024), scores_lds(16), stream, p);
    if (!fused) hipLaunchKernelGGL(bwd_dq_kernel<F16>, dim3((unsigned)(items * dq_parts)), dim3(64), 0, stream, p);
    const dim3 tiles((unsigned)((p.bands * ((p.D + 63) / 64) * p.shares * p.B * p.G + 7) / 8 * 8));
    hipLaunchKernelGGL(bwd_dkv_kernel<F16>, tiles, dim3(kDkvThreads), dkv_lds, stream, p);
    if (p.shares > 1) {
      const size_t n = (size_t)p.B * p.Skv * p.G * p.D / 4;
      hipLaunchKernelGGL(bwd_sum_kernel, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads), 0, stream, p);
    }
    CM_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

}  // namespace

bool sparse_mla_bwd_split_supports(const cppmega_mi355_sparse_mla_bwd_args_t& a) {
  const bool half = (a.q_dtype == CPPMEGA_MI355_BF16 || a.q_dtype == CPPMEGA_MI355_F16) && a.kv_dtype == a.q_dtype && a.d_out_dtype == a.q_dtype;
  if (!half || a.d_qk % 32 != 0 || a.d_v % 32 != 0 || a.d_qk > kBlocks * 64 || a.topk < 1 || a.topk > 2048) return false;
  if (a.batch < 1 || a.seq_q < 1 || a.seq_kv < 1 || a.seq_kv > 64 * 1024 || (long long)a.batch * a.kv_groups > 65535) return false;
  // A step costs the same for one key of a band as for sixteen, and the atomics the same for each key.  Measured at 64, 300 and 1000
  // queries over 1500 .. 60000 keys, time with the atomics over this path's by keys per 150 keys of the cache: up to 16 heads half a
  // key 0.7 .. 1.2, one 0.7 .. 1.4 (below one for 64 queries of up to 8000 keys and for 1000 of 20000), one and a half 0.7 .. 1.6; with more
  // heads, which that kernel adds up before its atomics, two 0.6 .. 1.6, three 0.7 .. 1.7 (below one for 64 queries of up to 4000 keys and
  // for 300 and 1000 of 20000), four 0.9 .. 1.7.
  const long long bands = ((long long)a.seq_kv + 149) / 150;
  if (bands * (a.heads / a.kv_groups > kHeads ? 3 : 1) > a.topk) return false;
  if ((long long)a.batch * a.seq_q * a.heads * ((a.d_qk + 143) / 144) > 0x7fffffffLL) return false;
  const Plan l = make_plan(a);
  // offsets into a slab are 32 bits, and so are the places of steps times 64
  return l.slab_bytes < 0x7fffffffu && (unsigned long long)a.batch * a.kv_groups * l.ns * l.list_steps < (1u << 26);
}

size_t sparse_mla_bwd_split_workspace_bytes(const cppmega_mi355_sparse_mla_bwd_args_t& a) { return make_plan(a).bytes; }

// dkv is written, or added to when clear_dkv is off: no clearing kernel in front.
int sparse_mla_bwd_split_launch(const cppmega_mi355_sparse_mla_bwd_args_t& a, hipStream_t stream) {
  const Plan l = make_plan(a);
  char* ws = static_cast<char*>(a.workspace);
  SplitParams p;
  p.q = static_cast<const unsigned short*>(a.q); p.kv = static_cast<const unsigned short*>(a.kv);
  p.d_out = static_cast<const unsigned short*>(a.d_out);
  p.indices = a.indices; p.sm_scale_dev = a.sm_scale_dev; p.dq = a.dq; p.dkv = a.dkv;
  p.keys = reinterpret_cast<int*>(ws + l.keys); p.starts = reinterpret_cast<int*>(ws + l.starts);
  p.band_steps = reinterpret_cast<int*>(ws + l.band_steps); p.steps = reinterpret_cast<i32x4*>(ws + l.steps);
  p.step_starts = reinterpret_cast<int*>(ws + l.step_starts); p.rows = reinterpret_cast<unsigned char*>(ws + l.rows);
  p.list_steps = (int)l.list_steps; p.dead_step = (unsigned)((size_t)a.batch * a.kv_groups * l.ns * l.list_steps * 64);
  p.planes = ws + l.planes; p.by_channel = reinterpret_cast<unsigned short*>(ws + l.by_channel);
  p.part = reinterpret_cast<float*>(ws + l.part);
  p.dq_dtype = a.dq_dtype; p.index_dtype = a.index_dtype;
  p.B = a.batch; p.S = a.seq_q; p.H = a.heads; p.G = a.kv_groups; p.Skv = a.seq_kv; p.topk = a.topk; p.D = a.d_qk; p.d_v = a.d_v;
  p.channels = (a.d_qk + 63) / 64 * 64;
  p.chunks = l.chunks; p.stride = l.stride; p.bands = l.bands; p.band_keys = l.band_keys;
  p.sm_scale = a.sm_scale;
  return a.q_dtype == CPPMEGA_MI355_F16 ? run<true>(p, l, a.clear_dkv != 0, stream) : run<false>(p, l, a.clear_dkv != 0, stream);
}

}  // namespace cm
