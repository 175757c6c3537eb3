// Sparse MLA forward by chunks of 16 heads on the matrix cores (gfx950), d_v = 512: KV groups of up to 16 heads, and few queries of more.
//
// Rows served: bf16 or float16 queries of 576 = 512 latent + 64 rope channels over key rows of the same type (packed, or a
// latent and a rope part); bf16 queries over e4m3 latent rows with fp32 scales (per 128 / 256 / 512 channels, per row, or
// none) and a bf16 rope tail; queries and key rows of 576 e4m3 codes with one fp32 scale each, or with E8M0 bytes per 32
// channels, over a bf16 copy in the workspace.
//
// The producer/consumer kernels (sparse_mla_latent.hip, sparse_mla_rows16.hip) share a tile of keys among 64 or 32 heads;
// with 16 most of their products are for heads that are not there, and a tile still takes 0.85 .. 1.25 us.  Here a
// wavefront has all heads, and the keys are what the four of a workgroup divide: each takes every fourth tile of 32 keys,
// with its own running maximum, and nobody waits for another one before the sums meet in LDS at the end.
//   S^T = K.Q^T (16x16x32): keys as rows, heads as columns, Q^T in registers.  A lane ends up with keys 4 kg .. 4 kg + 3
//   of both sub-tiles (16 keys) of its head: exactly the eight it needs as B operand of O^T = V^T.P^T when the contraction
//   runs over them in that order, so probabilities never leave the registers; V^T comes by transposing LDS reads in the
//   same order.  8-bit rows are converted (exactly) on their way out of LDS.
// A tile's rows come through registers, whole rows of neighbouring lanes, a tile ahead; a wavefront has the 512
// registers of a SIMD to itself.  Piece c (16 bytes) of row r stands at place c ^ fold: operand reads (16 rows, one
// piece) and transposing reads spread over the banks.
//
// Bound: a wavefront's own chain, alone on its SIMD.  Counters, 300 x 2048 16-bit rows / 700 x 1024 latent rows: it issues in 51 /
// 58 % of its time (vector 23 / 43 %: 8-bit rows are converted), waits for data in 31 / 34 %; the matrix cores are busy for 15 /
// 13 %, the LDS for 35 / 20 % of a workgroup's time, without a bank conflict.  Four tiles of 128 keys took 3.4 .. 5 us before.
// Measured (16 heads over 4096 keys; before -> here): 300 queries x 2048 keys: 16-bit rows 104 -> 82 us, latent 159 -> 92,
// codes 147 -> 85; 100 x 800 of 16 bits 24.7 -> 22.0, 100 x 512 latent 26.4 -> 18.8, codes 23.7 -> 17.0; one query x 2048 latent keys (splits) 20.3 -> 15.5.
// Error against float64 (rms, here over before, 64 x 512 .. 300 x 1000, scores of a deviation of 1, 2.9 and 7): output of 16-bit rows
// 0.72 .. 0.96, of 8-bit ones 0.93 .. 1.00; lse 0.92 .. 1.02.
// Operand reads are requested eight ahead of their products: with a wait for each (as the compiler orders them by itself)
// 700 queries x 1024 latent keys took 123 us, 84 so.

#include "sparse_mla_common.h"
#include "mfma_util.h"

namespace cm {

namespace {

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((ext_vector_type(4))) unsigned u4;

constexpr int kLat = 512, kRope = 64, kDqk = kLat + kRope;
constexpr int kTK = 32;                         // keys of a tile
constexpr int kWaves = 4;
constexpr float kLazy = 8.0f;                   // move a running maximum only when it grows by > 2^8

enum Rows { kRows16, kLatent, kCodes };

__device__ __forceinline__ int fold16(int r) { return ((r & 3) << 2) | (-(r >> 2) & 3); }
// 16-byte pieces of 8-bit rows: an operand read takes one piece of 16 rows, a transposing read one of rows 4 kg .. 4 kg + 3
// of both sub-tiles
__device__ __forceinline__ int fold8(int r) { return (r & 15) ^ ((r >> 1) & 8); }
__device__ __forceinline__ int fold_rope(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int fold_tail(int r) { return -(r >> 2) & 3; }

// bytes of a wavefront's tile in LDS: rows, the rope part (code rows: the last 64 codes), scales
template <int KIND> constexpr int kRowBytes = KIND == kRows16 ? 2 * kLat : kLat;
template <int KIND> constexpr int kTailBytes = KIND == kCodes ? kRope : 2 * kRope;
template <int KIND> constexpr int kTailOff = kTK * kRowBytes<KIND>;
template <int KIND> constexpr int kScaleOff = kTailOff<KIND> + kTK * kTailBytes<KIND>;
template <int KIND> constexpr int kTileBytes = kScaleOff<KIND> + (KIND == kRows16 ? 0 : kTK * 16);
constexpr int kMeetBytes = kWaves * 32 * 64 * 16;       // the wavefronts' sums
template <int KIND> constexpr int kSmem = (kWaves * kTileBytes<KIND> > kMeetBytes ? kWaves * kTileBytes<KIND> : kMeetBytes) + kWaves * 16 * 2 * 4;

// NBLK: fp32 scales per key row (1, 2 or 4); 0: none are given
template <int KIND, int NBLK, bool F16>
__global__ __launch_bounds__(kWaves * 64, 1) void sparse_mla_few_kernel(const MlaParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int nblk = NBLK ? NBLK : 1;
  const int tid = (int)threadIdx.x, lane = tid & 63, n = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* const tile = smem + wave * kTileBytes<KIND>;
  float* const stats = reinterpret_cast<float*>(smem + kSmem<KIND> - kWaves * 16 * 2 * 4);      // [wave][16 heads][max, sum]

  // which (query, KV group, split, 16 heads of the group); several queries per sequence: the last ones, with the longest causal
  // lists, first
  const unsigned chunks = (unsigned)(p.heads_per_group + 15) / 16u;
  unsigned id = p.S > 1 ? gridDim.x - 1u - blockIdx.x : blockIdx.x;
  if (chunks > 1) {                                       // the workgroups of one list in one XCD (launches go round the eight): each takes a run of them
    const unsigned q = gridDim.x >> 3, r = gridDim.x & 7, xcd = blockIdx.x & 7;
    id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (blockIdx.x >> 3);
  }
  const unsigned unit = id / chunks;
  const int chunk = (int)(id - unit * chunks);
  const unsigned qg = unit / (unsigned)p.num_splits;
  const int split = (int)(unit - qg * (unsigned)p.num_splits);
  const unsigned bs32 = qg / (unsigned)p.G;
  const int g = (int)(qg - bs32 * (unsigned)p.G), b = (int)(bs32 / (unsigned)p.S);
  const size_t bs = bs32;
  const int head0 = g * p.heads_per_group + 16 * chunk, heads_here = min(16, p.heads_per_group - 16 * chunk);
  const size_t idx_base = (bs * p.G + g) * (size_t)p.topk;
  const int key_begin = split * p.keys_per_split, key_end = min(p.topk, key_begin + p.keys_per_split);
  const int n_tiles = max(0, (key_end - key_begin + kTK - 1) / kTK);
  const float sm_scale = mla_sm_scale(p);

  // ---- a tile's keys: lane l % 32 has list entry l % 32 of it; -1 where there is none.  (Both halves of an entry are
  //      fetched, or the one twice: a branch on the type would wait for them at once.) ----
  const bool wide = p.index_dtype == CPPMEGA_MI355_I64;
  const int* const list = (const int*)p.indices + (wide ? 2 * idx_base : idx_base);
  struct Entry { int lo, hi; };
  auto entry_of = [&](int t) {
    const int i = min(key_begin + t * kTK + (lane & 31), p.topk - 1);
    const int* const at = list + (wide ? 2 * (size_t)i : (size_t)i);
    return Entry{at[0], at[wide ? 1 : 0]};
  };
  auto key_of = [&](int t, const Entry& e) {
    return key_begin + t * kTK + (lane & 31) < key_end && (unsigned)e.lo < (unsigned)p.Skv && (!wide || e.hi == 0) ? e.lo : -1;
  };
  // ---- its rows, whole rows of neighbouring lanes, into registers ----
  const size_t group_row0 = (size_t)b * p.Skv_pitch * p.G + g;
  const bool packed = KIND == kRows16 && p.rope_dim == 0;
  const unsigned row_pitch = KIND == kRows16 ? (packed ? 2 * kDqk : 2 * kLat) : (KIND == kCodes ? kDqk : kLat);
  const unsigned char* const rows = (const unsigned char*)p.kv + group_row0 * row_pitch;
  const unsigned char* const tails = KIND == kCodes ? rows + kLat : packed ? rows + 2 * kLat : (const unsigned char*)p.rope + group_row0 * (2 * kRope);
  // (a batch's rows are below 2^32 bytes from its first)
  const unsigned row_step = (unsigned)p.G * row_pitch, tail_step = KIND == kCodes || packed ? row_step : (unsigned)p.G * (2 * kRope);
  const __amdgpu_buffer_rsrc_t row_buf = __builtin_amdgcn_make_buffer_rsrc((void*)rows, 0, -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t tail_buf = __builtin_amdgcn_make_buffer_rsrc((void*)tails, 0, -1, 0x00020000);
  constexpr int kLanes = kRowBytes<KIND> / 16, kPer = 64 / kLanes, kRowLoads = kTK / kPer;        // lanes to a row, rows to a load
  constexpr int kTailLanes = kTailBytes<KIND> / 16, kTailPer = 64 / kTailLanes, kTailLoads = kTK / kTailPer;
  constexpr int kScaleLoads = KIND != kRows16 && NBLK ? (kTK * nblk + 63) / 64 : 0;
  u4 row_regs[kRowLoads], tail_regs[kTailLoads];
  float scale_regs[2];
  // (a skipped key fetches a valid one's row of the same tile: its probability is zero, but a row that nobody selected
  // may hold NaN or infinity)
  auto request = [&](int keys, unsigned valid) {
    const int spare = __builtin_amdgcn_readlane(keys, __builtin_ctz(valid));
    keys = keys >= 0 ? keys : spare;
    unsigned tail_key[kTailLoads], scale_key[2];
#pragma unroll
    for (int i = 0; i < kTailLoads; ++i) tail_key[i] = (unsigned)__shfl(keys, i * kTailPer + lane / kTailLanes, 64);
#pragma unroll
    for (int i = 0; i < kScaleLoads; ++i) scale_key[i] = (unsigned)__shfl(keys, min(i * 64 + lane, kTK * nblk - 1) / nblk, 64);
    const unsigned offs = (unsigned)keys * row_step;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i) {
      const unsigned at = 16 * (unsigned)(lane % kLanes);
      if (kPer == 1) {
        row_regs[i] = __builtin_amdgcn_raw_buffer_load_b128(row_buf, (int)at, __builtin_amdgcn_readlane((int)offs, i), 0);
      } else {
        const int even = __builtin_amdgcn_readlane((int)offs, 2 * i), odd = __builtin_amdgcn_readlane((int)offs, 2 * i + 1);
        row_regs[i] = __builtin_amdgcn_raw_buffer_load_b128(row_buf, (int)(at + (unsigned)(lane < 32 ? even : odd)), 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < kTailLoads; ++i)
      tail_regs[i] = __builtin_amdgcn_raw_buffer_load_b128(tail_buf, (int)(tail_key[i] * tail_step + 16 * (unsigned)(lane % kTailLanes)), 0, 0);
#pragma unroll
    for (int i = 0; i < kScaleLoads; ++i)
      scale_regs[i] = ((const float*)p.kv_scale)[(group_row0 + (size_t)scale_key[i] * p.G) * nblk + min(i * 64 + lane, kTK * nblk - 1) % nblk];
  };
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i) {
      const int r = i * kPer + lane / kLanes, c = lane % kLanes;
      *reinterpret_cast<u4*>(tile + r * kRowBytes<KIND> + ((c ^ (KIND == kRows16 ? fold16(r & 15) : fold8(r))) * 16)) = row_regs[i];
    }
#pragma unroll
    for (int i = 0; i < kTailLoads; ++i) {
      const int r = i * kTailPer + lane / kTailLanes, c = lane % kTailLanes;
      *reinterpret_cast<u4*>(tile + kTailOff<KIND> + r * kTailBytes<KIND> + ((c ^ (KIND == kCodes ? fold_tail(r & 15) : fold_rope(r & 15))) * 16)) = tail_regs[i];
    }
    if (KIND != kRows16)
#pragma unroll
      for (int i = 0; i < (kTK * nblk + 63) / 64; ++i)
        if (i * 64 + lane < kTK * nblk) reinterpret_cast<float*>(tile + kScaleOff<KIND>)[i * 64 + lane] = NBLK ? scale_regs[i] : 1.0f;
  };
  // the next tile with a valid key: its keys and which count
  int t_next = wave, keys_next = -1;
  unsigned valid_next = 0;
  Entry ahead = entry_of(min(t_next, max(n_tiles - 1, 0)));
  auto find = [&]() {
    valid_next = 0;
    while (t_next < n_tiles) {
      keys_next = key_of(t_next, ahead);
      valid_next = (unsigned)__ballot(keys_next >= 0);
      t_next += kWaves;
      ahead = entry_of(min(t_next, n_tiles - 1));
      if (valid_next) return;
    }
  };

  // ---- Q^T: lane (head n, kg).  16-bit keys: step ks holds channels 32 ks + 8 kg .. + 7.  8-bit keys: a lane's 16 codes
  //      are channels 64 s + 16 kg .. + 15 and serve the steps 2 s and 2 s + 1; a rope tail is in the order of 16-bit keys ----
  bf16x8 qf[18];
  {
    const int h = n < heads_here ? n : 0;                 // (heads past the end repeat head 0 and are never stored)
    const size_t q_row = (bs * p.H + head0 + h) * (size_t)kDqk;
#pragma unroll
    for (int ks = 0; ks < 18; ++ks) {
      const bool split_order = KIND == kCodes || (KIND == kLatent && ks < 16);
      const int ch = split_order ? 64 * (ks >> 1) + 16 * kg + 8 * (ks & 1) : 32 * ks + 8 * kg;
      if (KIND == kCodes) {
        const uint2 c = *reinterpret_cast<const uint2*>((const unsigned char*)p.q + q_row + ch);
        qf[ks] = cvt8(c.x, c.y);
      } else {
        qf[ks] = *reinterpret_cast<const bf16x8*>((const unsigned short*)p.q + q_row + ch);
      }
    }
  }
  float q_scale = 1.0f;
  if (KIND == kCodes) q_scale = ((const float*)p.q_scale)[bs * p.H + head0 + (n < heads_here ? n : 0)];
  const float qk_scale = sm_scale * kLog2e * q_scale;

  f32x4 o[32];                                            // channels 16 c + 4 kg + v of head n
#pragma unroll
  for (int c = 0; c < 32; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.0f;                  // base-2 reference of head n, this lane's share of its denominator

  // transposing reads: lane t of a group of 16 points at the rows of the group's eight keys 16 (j / 4) + 4 kg + j % 4
  const unsigned char* v_at[2];
  int v_fold[2];
  if (KIND == kRows16) {
#pragma unroll
    for (int sj = 0; sj < 2; ++sj) {                      // four keys of a sub-tile, 8 bytes each
      const int r = 4 * kg + (n >> 2);
      v_at[sj] = tile + (16 * sj + r) * kRowBytes<KIND> + (n & 1) * 8;
      v_fold[sj] = fold16(r) ^ ((n >> 1) & 1);
    }
  } else {
    const int j = n >> 1, r = 4 * kg + (j & 3);
    v_at[0] = tile + (16 * (j >> 2) + r) * kRowBytes<KIND> + (n & 1) * 8;
    v_fold[0] = fold8(16 * (j >> 2) + r);
    v_at[1] = v_at[0];
    v_fold[1] = v_fold[0];
  }

  find();
  if (valid_next) request(keys_next, valid_next);
  while (valid_next) {
    const unsigned valid = valid_next;
    put();
    __builtin_amdgcn_wave_barrier();
    find();
    if (valid_next) request(keys_next, valid_next);       // (uniform)

    // ---- scores: this lane holds head n, keys 16 sj + 4 kg + i ----
    float ks[2][4][nblk];
    if (KIND != kRows16)
#pragma unroll
      for (int sj = 0; sj < 2; ++sj)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < nblk; ++c) ks[sj][i][c] = reinterpret_cast<const float*>(tile + kScaleOff<KIND>)[(16 * sj + 4 * kg + i) * nblk + c];
    f32x4 st[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    // operand pieces are requested kDeep ahead of their products (in the order written: with a wait for each, a tile of
    // 16-bit rows took 11000 clocks)
    constexpr int kSteps = KIND == kRows16 ? 36 : 16, kTailSteps = KIND == kCodes ? 2 : 4, kDeep = 8;
    uint4 piece[kDeep], tail[kTailSteps];
    auto fetch = [&](int i) {                             // step i: piece i / 2 of the rows of sub-tile i % 2
      const int s = i >> 1, r = 16 * (i & 1) + n;
      if (KIND == kRows16 && s >= 16)
        return *reinterpret_cast<const uint4*>(tile + kTailOff<KIND> + r * kTailBytes<KIND> + (((4 * (s - 16) + kg) ^ fold_rope(n)) * 16));
      return *reinterpret_cast<const uint4*>(tile + r * kRowBytes<KIND> + (((4 * s + kg) ^ (KIND == kRows16 ? fold16(n) : fold8(r))) * 16));
    };
    if constexpr (KIND != kRows16)
#pragma unroll
      for (int i = 0; i < kTailSteps; ++i) {
        const int r = 16 * (i & 1) + n, c = 4 * (i >> 1) + kg;
        tail[i] = *reinterpret_cast<const uint4*>(tile + kTailOff<KIND> + r * kTailBytes<KIND> + ((c ^ (KIND == kCodes ? fold_tail(n) : fold_rope(n))) * 16));
      }
#pragma unroll
    for (int i = 0; i < kDeep; ++i) piece[i] = fetch(i);
    __builtin_amdgcn_sched_barrier(0);
    // Latent rows: the rope part first, then every 128 channels accumulated from zero and added times their keys' scales, however
    // few those are.  With a chain through all channels, rounded 18 times at the size of the score, lse was off by 1.2 times as
    // much at scores of a deviation of 2.9 and by 1.7 at 7.  (Code rows: one chain, the tail last, then the scale; it made no difference.)
    f32x4 part[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    if constexpr (KIND == kLatent)
#pragma unroll
      for (int i = 0; i < 4; ++i) st[i & 1] = mm<false>(__builtin_bit_cast(bf16x8, tail[i]), qf[16 + (i >> 1)], st[i & 1]);
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const uint4 w = piece[i % kDeep];
      const int sj = i & 1, s = i >> 1;
      if constexpr (KIND == kRows16) {
        st[sj] = mm<F16>(__builtin_bit_cast(bf16x8, w), qf[s], st[sj]);
      } else {
        part[sj] = mm<false>(cvt8(w.x, w.y), qf[2 * s], part[sj]);
        part[sj] = mm<false>(cvt8(w.z, w.w), qf[2 * s + 1], part[sj]);
      }
      if (i + kDeep < kSteps) piece[i % kDeep] = fetch(i + kDeep);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (KIND != kRows16) {
        if (KIND == kCodes && i >= kSteps - 2) {
          part[sj] = mm<false>(cvt8(tail[sj].x, tail[sj].y), qf[16], part[sj]);
          part[sj] = mm<false>(cvt8(tail[sj].z, tail[sj].w), qf[17], part[sj]);
        }
        if (KIND == kCodes ? s == 7 : (s & 1) != 0) {
#pragma unroll
          for (int e = 0; e < 4; ++e) st[sj][e] = __builtin_fmaf(ks[sj][e][s * nblk / 8], part[sj][e], st[sj][e]);
          part[sj] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
    // V^T of the first blocks, during the softmax
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    constexpr int kDeepV = 8;
    u32x2 vt[kDeepV][KIND == kRows16 ? 2 : 1];
    auto fetch_v = [&](int blk) {
      if constexpr (KIND == kRows16) {
#pragma unroll
        for (int sj = 0; sj < 2; ++sj)
          vt[blk % kDeepV][sj] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(v_at[sj] + (((2 * blk) ^ v_fold[sj]) * 16))));
      } else {
        vt[blk % kDeepV][0] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) i32x2*)(v_at[0] + ((blk ^ v_fold[0]) * 16))));
      }
    };
#pragma unroll
    for (int blk = 0; blk < kDeepV; ++blk) fetch_v(blk);
    __builtin_amdgcn_sched_barrier(0);
    // ---- softmax ----
    float mx = -INFINITY;
    auto counts = [&](int e) { return ((valid >> (16 * (e >> 2) + 4 * kg + (e & 3))) & 1u) != 0; };
    if (valid == 0xffffffffu) {                           // (uniform, and the rule)
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, st[e >> 2][e & 3] * qk_scale);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, counts(e) ? st[e >> 2][e & 3] * qk_scale : -INFINITY);
    }
    mx = max_rows(mx);
    const bool grow = mx > m_run + kLazy || (m_run == -INFINITY && mx > -INFINITY);
    if (__ballot(grow) != 0ull) {                         // (rare behind the first tile)
      float fac = 1.0f;
      if (grow) {
        fac = m_run == -INFINITY ? 1.0f : fast_exp2(m_run - mx);        // (the sums of a head without a reference are zero)
        l_run *= fac;
        m_run = mx;
      }
#pragma unroll
      for (int c = 0; c < 32; ++c) o[c] *= fac;
    }
    const float neg_m = m_run > -INFINITY ? -m_run : 0.0f;
    float pr[8];
    // (scaled inside the multiply-add: a product by itself is rounded at the size of the score)
#pragma unroll
    for (int e = 0; e < 8; ++e) pr[e] = fast_exp2(__builtin_fmaf(st[e >> 2][e & 3], qk_scale, neg_m));
    if (valid != 0xffffffffu)
#pragma unroll
      for (int e = 0; e < 8; ++e) pr[e] = counts(e) ? pr[e] : 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) l_run += pr[e];
    // ---- O^T += V^T.P^T ----
#pragma unroll
    for (int c = 0; c < nblk; ++c) {
      float ps[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) ps[e] = KIND == kRows16 ? pr[e] : pr[e] * ks[e >> 2][e & 3][c];
      const bf16x8 pb = __builtin_bit_cast(bf16x8, F16 ? make_uint4(pack_f16(ps[0], ps[1]), pack_f16(ps[2], ps[3]), pack_f16(ps[4], ps[5]), pack_f16(ps[6], ps[7]))
                                                       : make_uint4(pack_bf16(ps[0], ps[1]), pack_bf16(ps[2], ps[3]), pack_bf16(ps[4], ps[5]), pack_bf16(ps[6], ps[7])));
#pragma unroll
      for (int blk = c * (32 / nblk); blk < (c + 1) * (32 / nblk); ++blk) {
        bf16x8 v;
        const u32x2* const w = vt[blk % kDeepV];
        if constexpr (KIND == kRows16) v = __builtin_bit_cast(bf16x8, make_uint4(w[0][0], w[0][1], w[1][0], w[1][1]));
        else v = cvt8(w[0][0], w[0][1]);
        o[blk] = mm<F16>(v, pb, o[blk]);
        if (blk + kDeepV < 32) fetch_v(blk + kDeepV);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }

  // ---- the four wavefronts' sums ----
  l_run += xor16(l_run);
  l_run += xor32(l_run);
  if (lane < 16) {
    stats[(wave * 16 + n) * 2] = m_run;
    stats[(wave * 16 + n) * 2 + 1] = l_run;
  }
  __syncthreads();                                        // (and the tiles are read)
  float m_all = -INFINITY, l_all = 0.0f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) m_all = fmaxf(m_all, stats[(w * 16 + n) * 2]);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float m = stats[(w * 16 + n) * 2];
    l_all += m > -INFINITY ? stats[(w * 16 + n) * 2 + 1] * fast_exp2(m - m_all) : 0.0f;
  }
  const float own = m_run > -INFINITY ? fast_exp2(m_run - m_all) : 0.0f;
  f32x4* const meet = reinterpret_cast<f32x4*>(smem);     // [wave][block of 16 channels][lane]
  const int working = min(kWaves, n_tiles);               // (the first have the tiles)
  if (wave < working)
#pragma unroll
    for (int c = 0; c < 32; ++c) meet[(wave * 32 + c) * 64 + lane] = o[c] * own;
  __syncthreads();
  float out_scale = 1.0f, lse_val = 0.0f;
  const bool direct = p.num_splits == 1;
  if (direct) {
    float m_fin = m_all, l_fin = l_all;
    if (mla_has_sinks(p) && n < heads_here) {
      const float sk = p.sinks[head0 + n] * kLog2e, m2 = fmaxf(m_fin, sk);
      const float keep = (m_fin == -INFINITY) ? 0.0f : exp2f(m_fin - m2);
      l_fin = l_fin * keep + exp2f(sk - m2);
      out_scale = keep;
      m_fin = m2;
    }
    if (l_fin > 0.0f) {
      out_scale = out_scale / l_fin;
      lse_val = (m_fin + log2f(l_fin)) * kLn2;
    } else {
      out_scale = 0.0f;
    }
  }
  // (a partial block holds 32 heads, two workgroups')
  const unsigned blocks32 = (chunks + 1) / 2;
  const size_t part_block = ((size_t)qg * blocks32 + chunk / 2) * p.num_splits + split, part_blocks = (size_t)p.B * p.S * p.G * blocks32 * p.num_splits;
  const int part_head = 16 * (chunk & 1) + n;
  // this wavefront finishes blocks 8 wave .. 8 wave + 7 (128 channels)
  f32x4 sums[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int w = 0; w < working; ++w)
#pragma unroll
    for (int i = 0; i < 8; ++i) sums[i] += meet[(w * 32 + 8 * wave + i) * 64 + lane];
  if (!direct) {
    // as sparse_mla_latent_combine_kernel takes it: channels 128 wave + 32 dvb + 8 j + 4 half .. of head n
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int dvb = i >> 1, j = 2 * (i & 1) + (kg >> 1), half = kg & 1;
      float* blk = (float*)p.workspace + part_block * (size_t)kMlaPartFloats + ((size_t)(wave * 8) * 64 + half * 32 + part_head) * 8;
      *reinterpret_cast<f32x4*>(blk + (size_t)(dvb * 2 + (j >> 1)) * 512 + (j & 1) * 4) = sums[i];
    }
  } else if (n < heads_here) {
    const size_t off = (bs * p.H + head0 + n) * (size_t)kLat + 128 * wave + 4 * kg;
#pragma unroll
    for (int i = 0; i < 8; ++i) sums[i] *= out_scale;
    if ((uintptr_t)p.out & 15) {                          // (uniform; not part of the choice of a plan: scratch is asked for before there is an output)
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) store_as(p.out, off + 16 * i + e, p.out_dtype, sums[i][e]);
    } else if (p.out_dtype == CPPMEGA_MI355_F32) {
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>((float*)p.out + off + 16 * i) = sums[i];
    } else {
      const bool bf = p.out_dtype == CPPMEGA_MI355_BF16;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        *reinterpret_cast<uint2*>((unsigned short*)p.out + off + 16 * i) =
            make_uint2(bf ? pack_bf16(sums[i][0], sums[i][1]) : pack_f16(sums[i][0], sums[i][1]), bf ? pack_bf16(sums[i][2], sums[i][3]) : pack_f16(sums[i][2], sums[i][3]));
    }
  }
  if (wave == 0 && lane < 16) {
    if (!direct) {
      float* ml = (float*)p.workspace + part_blocks * (size_t)kMlaPartFloats + (part_block * 32 + part_head) * 2;
      ml[0] = m_all;
      ml[1] = l_all;
    } else if (n < heads_here && p.lse) {
      p.lse[bs * p.H + head0 + n] = lse_val;
    }
  }
}

template <int KIND, int NBLK, bool F16>
int launch_as(const MlaParams& p, hipStream_t stream) {
  void (*kernel)(MlaParams) = sparse_mla_few_kernel<KIND, NBLK, F16>;
  CM_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kSmem<KIND>));
  hipLaunchKernelGGL(kernel, dim3((unsigned)((size_t)p.B * p.S * p.G * ((p.heads_per_group + 15) / 16) * p.num_splits)), dim3(kWaves * 64), kSmem<KIND>, stream, p);
  CM_HIP_CHECK(hipGetLastError());
  return p.num_splits > 1 ? sparse_mla_combine_f32(p, stream) : 0;
}

}  // namespace

namespace {
// The number of splits with the least modelled time: rounds of 256 workgroups, each with its start and end and the
// tiles that one of its four wavefronts has, then the merging kernel and its traffic.  Fitted to 147 shapes (three kinds
// of rows, 1 .. 300 queries, 128 .. 2048 keys, up to 16 splits): 0.5 % from the best number in the mean, 8 % at most.
// `units`: queries, KV groups and chunks of 16 heads.
double few_splits(long long units, int topk, int* splits, int* keys_per_split) {
  const int tiles = (topk + kTK - 1) / kTK;
  double best = 0.0;
  *splits = 0;
  for (int s = 1; s <= 16; ++s) {
    const int per = (tiles + s - 1) / s, used = (tiles + per - 1) / per;
    double us = (double)((units * used + 255) / 256) * (4.0 + 2.1 * ((per + kWaves - 1) / kWaves));
    if (used > 1) us += 2.0 + 0.2 * used + (double)units * used * kMlaPartFloats * 4 / 4e6;
    if (*splits == 0 || us < best) {
      best = us;
      *splits = used;
      *keys_per_split = per * kTK;
    }
  }
  return best;
}
long long units_of(const MlaParams& p) { return (long long)p.B * p.S * p.G * ((p.heads_per_group + 15) / 16); }
}  // namespace

bool sparse_mla_few_supported(const MlaParams& p) {
  if (p.d_qk != kDqk || p.d_v != kLat) return false;
  const long long units = units_of(p);
  if (units * 16 > 0x7fffffffll) return false;
  const bool of_16_bits = sparse_mla_rows16_supported(p);
  if (of_16_bits && sparse_mla_e8m0_copy_bytes(p) > ((size_t)1 << 30)) return false;
  if (p.heads_per_group > 16) {
    // More heads: few queries leave CUs idle where 64 heads share a workgroup, chunks of 16 fill them (4 queries x 128 heads, before /
    // here: 128 keys of 16-bit rows 12.4 / 10.2 us, 512 19.2 / 15.3, 2048 26.8 / 20.2, codes 26.5 / 20.0, E8M0 rows 32.2 / 27.0; 64 queries x
    // 64 heads x 512 25.1 / 18.4).  A unit takes about 1.4 times what its model says beside that of the other kernel, 1.5 over the
    // copy of E8M0 rows, whose queries cost 0.35 ns a row: of 354 shapes (64 and 128 heads, 1 .. 500 queries, 64 .. 2048 keys, three kinds of rows) those that
    // pass gain 1.17 x in the mean and none loses; one round more of workgroups (96 queries x 128 heads x 512 26.9 / 51.0) and long lists
    // of 24 queries on (24 x 64 x 2048 26.9 / 32.1) stay where they were.  Latent rows: no gain at 1 or 2 queries, slower from 4 on.
    if (p.no_few || (!of_16_bits && p.q_dtype != CPPMEGA_MI355_E4M3)) return false;
    int splits, keys;
    MlaParams other = p;
    double other_us;
    if (of_16_bits) other_us = sparse_mla_rows16_plan(other);
    else if (sparse_mla_latent_supported(p)) other_us = sparse_mla_latent_plan(other);
    else return false;
    const bool copied = of_16_bits && p.q_dtype == CPPMEGA_MI355_E4M3;
    return (copied ? 1.5 : 1.4) * few_splits(units, p.topk, &splits, &keys) + (copied ? 0.35e-3 * p.B * p.S * p.H : 0.0) < other_us;
  }
  // 8-bit rows: at 64 keys as fast as the kernel for 64 heads (9.3 / 9.1 us latent, 7.9 / 8.2 codes, one query), from there on
  // faster.  16-bit rows: a wavefront's tile takes 2.1 us from first to last, so short lists and few queries
  // are better off with four wavefronts at one tile (32 x 320: 13.2 us there, 14.3 here; 4 x 2048: 15.9 / 16.1; 32 x 512: 15.2 / 14.9;
  // 8 x 2048: 17.6 / 16.8; 100 x 800: 26.1 / 23.2).  E8M0 rows, whose queries are copied too: 13 x 2048 25.5 / 22.4, 500 x 1100 70.5 / 64.5,
  // 118 x 1100 33.7 / 33.7, 903 x 1161 88.8 / 91.7, 500 x 728 38.1 / 43.2.
  if (of_16_bits && p.q_dtype == CPPMEGA_MI355_E4M3) return !p.no_few && p.topk >= 1280 && units * p.topk >= 16384;
  if (of_16_bits) return p.topk >= 512 && units * p.topk >= 16384;
  return sparse_mla_latent_supported(p);
}

void sparse_mla_few_plan(MlaParams& p) {
  p.few = 1;
  p.heads_per_wg = 32;                                    // (what the merging kernel takes a partial block for)
  few_splits(units_of(p), p.topk, &p.num_splits, &p.keys_per_split);
}

int sparse_mla_few_launch(const MlaParams& p, hipStream_t stream) {
  if (p.num_splits > 16) return fail(CPPMEGA_MI355_ERR_UNSUPPORTED, "sparse MLA: launch too large");
  if (sparse_mla_e8m0_copy_bytes(p)) {                      // queries and rows as the bfloat16 values they stand for
    MlaParams copy = p;
    const int rc = sparse_mla_e8m0_copy(copy, stream);
    return rc ? rc : launch_as<kRows16, 0, false>(copy, stream);
  }
  if (p.kv_dtype != CPPMEGA_MI355_E4M3)
    return p.q_dtype == CPPMEGA_MI355_F16 ? launch_as<kRows16, 0, true>(p, stream) : launch_as<kRows16, 0, false>(p, stream);
  if (p.q_dtype == CPPMEGA_MI355_E4M3) return launch_as<kCodes, 1, false>(p, stream);
  if (p.kv_scale_kind == CPPMEGA_MI355_SCALE_NONE) return launch_as<kLatent, 0, false>(p, stream);
  const int nblk = p.kv_scale_kind == CPPMEGA_MI355_SCALE_F32_BLOCK ? kLat / p.kv_scale_block : 1;
  return nblk == 4 ? launch_as<kLatent, 4, false>(p, stream) : nblk == 2 ? launch_as<kLatent, 2, false>(p, stream) : launch_as<kLatent, 1, false>(p, stream);
}

size_t sparse_mla_few_workspace_bytes(const MlaParams& p) {
  const size_t copy = sparse_mla_e8m0_copy_bytes(p);
  if (p.num_splits <= 1) return copy;
  // (8-bit rows of up to 16 heads: as much per split as the kernel for 64 heads asks for, so that scratch for the one serves the other)
  const size_t blocks = p.heads_per_group > 16 ? (p.heads_per_group + 31) / 32 : p.kv_dtype == CPPMEGA_MI355_E4M3 && !copy ? 2 : 1;
  return copy + (size_t)p.B * p.S * p.G * p.num_splits * blocks * (size_t)(kMlaPartFloats + 32 * 2) * sizeof(float);
}

}  // namespace cm
