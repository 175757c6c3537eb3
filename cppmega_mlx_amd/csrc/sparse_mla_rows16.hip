// Sparse MLA forward over 16-bit key rows on the matrix cores (gfx950), with the wavefronts of a
// workgroup split into score producers and value consumers.
//
// Shapes served: queries and key rows of 576 e4m3 codes with one E8M0 byte per 32 channels, and bf16 or float16
// queries of 576 = 512 latent + 64 rope channels over key rows of the same type, packed (576) or as latent rows of
// 512 plus a rope tail of 64; d_v = 512.
// A power of two times an e4m3 code is a bfloat16: E8M0 rows become bf16 rows in the workspace first (all of them, about
// 6 us for 16384), the query's codes on their way to operand order, and nothing is rounded.
//
// Measured against the kernel of sparse_mla_mfma.hip, bf16: 64 queries x 16 heads x 64 keys 33 -> 7.8 us (the whole
// call); 1000 queries x 2048 keys: 16 heads 573 -> 210 us, 64 heads 910 -> 304 us, 128 heads 953 -> 600 us (the
// products at the rate of a large matrix product: 457 us).  Of 73 shapes (1 .. 1000 queries, 64 .. 2048 keys) none
// was slower; 2.6x in the mean.  E8M0 rows, 128 heads: 1500 x 2048 of 16384 1726 -> 890 us, 30 x 256 64 -> 25 us; 45 shapes
// 2.4x in the mean.  What is left: 1.0 us per tile at 64 heads, where the products of a SIMD are 1088
// clocks, and about 8 us for a workgroup's start and end, which nothing overlaps: the ring fills the LDS of the CU.
//
// Workgroup = (query, KV group, chunk of 32 HB heads, key split), 8 wavefronts, key tiles of 32 rows in a
// ring of four LDS slots filled by the load unit (global_load_lds) three tiles ahead.  Two wavefronts
// share a SIMD: one producer and one consumer.
//
//   producers (wavefronts 0..3): producer p owns sub-tile p / 2 (16 keys) and heads 16 HB (p % 2) .. of the
//     chunk: S^T = K.Q^T on 16x16x32 products, Q^T in registers, a K fragment read from LDS serving HB head
//     groups.  (With a producer per 16 heads and all 32 keys the four of them read every tile four times:
//     200 KB of LDS per tile, more than the products take; this way 122 KB.)  The two producers of a
//     head group exchange their tile maxima through LDS at a barrier in the middle of the iteration, so that
//     both write probabilities relative to the same reference.
//   consumers (wavefronts 4..7): consumer c owns value channels 128c..128c+127 for all heads of the chunk:
//     O^T += V^T.P^T on 32x32x16 products, V^T fragments by transposing LDS reads of the same tile.  They
//     also issue the row loads.
//   pipeline  iteration t: producers: scores of tile t+1 | exchange | P of tile t+1; consumers: issue tile t+3,
//     first key step of the value product of tile t | second key step.
//
// LDS rows keep the order of memory, so a load instruction moves one row (64 lanes on neighbouring 16-byte
// pieces: a load whose lanes each point into another row moves a quarter of the bytes per clock); lane l of row r
// fetches piece l ^ fold(r), which spreads both the operand reads (16 rows, one piece each) and the transposing
// reads (4 rows, 4 pieces) over all banks.

#include "sparse_mla_common.h"
#include "mfma_util.h"

namespace cm {

namespace {

constexpr int kLat = 512;
constexpr int kRope = 64;
constexpr int kDqk = kLat + kRope;
constexpr int kTK = 32;                         // keys per tile
constexpr int kRing = 4;                        // latent slots
constexpr int kRopeRing = 3;                    // rope slots: a tile's is free one iteration earlier
constexpr int kAhead = 3;                       // tiles issued ahead of the value product
constexpr int kLatRow = kLat * 2;
constexpr int kLatSlot = kTK * kLatRow;         // 32768
constexpr int kRopeRow = kRope * 2;
constexpr int kRopeSlot = kTK * kRopeRow;       // 4096
constexpr int kMaxKeys = 2048;                  // keys of one split (their rows are staged in LDS)
constexpr int kKeyInts = kMaxKeys + kTK;
constexpr int kXPitch = 132;                    // floats per head row of the output transpose (128 + 4)
constexpr float kLazy = 8.0f;                   // move a running maximum only when it grows by > 2^8
constexpr int kLoads = 9;                       // load instructions of a tile per consumer

constexpr int kRopeOff = kRing * kLatSlot;                     // 131072
constexpr int kPOff = kRopeOff + kRopeRing * kRopeSlot;        // [parity][sub-tile][32-head block][64 lanes x 16 B]
constexpr int kFacOff = kPOff + 2 * 2 * 2 * 1024;              // [parity][64 heads] fp32
constexpr int kFlagOff = kFacOff + 2 * 64 * 4;                 // [parity][2 head halves] int
constexpr int kMaxOff = kFlagOff + 2 * 2 * 4;                  // [sub-tile][64 heads] fp32: maxima of the tile being produced
constexpr int kStatOff = kMaxOff + 2 * 64 * 4;                 // [sub-tile][64 heads][2] fp32
constexpr int kValidOff = kStatOff + 2 * 64 * 2 * 4;           // [tile] int: every key of the tile is valid
constexpr int kKeyOff = kValidOff + (kMaxKeys / kTK) * 4;
constexpr int kSmem = kKeyOff + kKeyInts * 4;
static_assert(kSmem <= 160 * 1024, "LDS budget");
static_assert(4 * 32 * kXPitch * 4 <= kRopeOff, "the output transpose reuses the ring");
constexpr int kQPitch = kDqk * 2 + 16;          // a staged query row
static_assert(64 * kQPitch <= (kRing - 1) * kLatSlot, "the query rows fit the slots behind the first tile");

// A bijection of a row's number within 16: rows 4j .. 4j+3 differ in its upper two bits (transposing reads), and the
// 16 rows, of which the load unit's groups take eight with piece q and eight with q ^ 1, meet on no bank.
__device__ __forceinline__ int fold(int r) { return ((r & 3) << 2) | (-(r >> 2) & 3); }
// The same for the 8 pieces of a rope row (two rows to a pass over the banks).
__device__ __forceinline__ int fold_rope(int r) { return ((r << 1) & 4) | (-(r >> 2) & 3); }

template <bool F16>
__device__ __forceinline__ void mfma_s(f32x4& acc, const bf16x8& a, const bf16x8& b) {
  if (F16) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
  else acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
template <bool F16>
__device__ __forceinline__ void mfma_o(f32x16& acc, const bf16x8& a, const bf16x8& b) {
  if (F16) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
  else acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}

// HB: 32-head blocks of the chunk (1 or 2)
// Q_E8: the queries are e4m3 codes with E8M0 scales
template <bool F16, int HB, bool Q_E8 = false>
__global__ __launch_bounds__(512, 2) void sparse_mla_rows16_kernel(const MlaParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int kHeadsWg = 32 * HB;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool producer = wave < 4;
  const int role = wave & 3;                    // producer p / consumer c

  // ---- which (query, KV group, head chunk, split): ids that are equal modulo 8 share an XCD and its L2, so
  //      every workgroup of one (query, KV group) gets such ids ----
  const unsigned chunks = (unsigned)(p.heads_per_group + kHeadsWg - 1) / (unsigned)kHeadsWg;
  const unsigned per_q = (unsigned)p.num_splits * chunks;
  const unsigned nq = (unsigned)p.B * (unsigned)p.S * (unsigned)p.G;
  const unsigned nq8 = nq & ~7u;
  unsigned qg;
  int chunk, split;
  {
    // (several queries per sequence: the last ones first - under a causal selection they hold the longest lists)
    const unsigned id = p.S > 1 ? gridDim.x - 1u - blockIdx.x : blockIdx.x;
    unsigned r;
    if (id < nq8 * per_q) {
      const unsigned slot = id >> 3, sq = slot / per_q;
      qg = sq * 8u + (id & 7u);
      r = slot - sq * per_q;
    } else {
      const unsigned rest = id - nq8 * per_q, rq = rest / per_q;
      qg = nq8 + rq;
      r = rest - rq * per_q;
    }
    split = (int)(r / chunks);
    chunk = (int)(r - (unsigned)split * chunks);
  }
  const unsigned bs32 = qg / (unsigned)p.G;       // b*S + s
  const int g = (int)(qg - bs32 * (unsigned)p.G);
  const size_t bs = bs32;
  const int b = (int)(bs32 / (unsigned)p.S);
  const int head0 = g * p.heads_per_group + chunk * kHeadsWg;
  const int heads_here = min(kHeadsWg, p.heads_per_group - chunk * kHeadsWg);
  const size_t idx_base = (bs * p.G + g) * (size_t)p.topk;
  const int key_begin = split * p.keys_per_split;
  const int key_end = min(p.topk, key_begin + p.keys_per_split);
  const int n_keys = max(0, key_end - key_begin);
  const int list_tiles = (n_keys + kTK - 1) / kTK;

  int* keys = reinterpret_cast<int*>(smem + kKeyOff);
  float* facbuf = reinterpret_cast<float*>(smem + kFacOff);
  int* flagbuf = reinterpret_cast<int*>(smem + kFlagOff);
  float* maxbuf = reinterpret_cast<float*>(smem + kMaxOff);
  float* stats = reinterpret_cast<float*>(smem + kStatOff);
  int* tvalid = reinterpret_cast<int*>(smem + kValidOff);

  // ---- cache rows of this split's keys -> LDS (-1 = skipped).  Every index word is requested before the first one is
  //      looked at; the producers put their query-row requests between the two halves ----
  int* last_valid = reinterpret_cast<int*>(stats);          // [8], one per wavefront
  constexpr int kRounds = kMaxKeys / 512;
  const bool wide = p.index_dtype == CPPMEGA_MI355_I64;
  const float qk_scale = mla_sm_scale(p) * kLog2e;
  int idx_lo[kRounds], idx_hi[kRounds];
  {
    const int* words = (const int*)p.indices;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      idx_lo[r] = 0; idx_hi[r] = 0;
      if (r * 512 < list_tiles * kTK) {           // (uniform)
        const size_t at = idx_base + (size_t)min(key_begin + tid + 512 * r, p.topk - 1);
        const size_t w0 = wide ? 2 * at : at;
        idx_lo[r] = words[w0];
        idx_hi[r] = words[w0 + (wide ? 1 : 0)];
      }
    }
  }
  auto stage_keys = [&]() {
    int mine = -1;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      if (r * 512 < list_tiles * kTK) {
        const int i = tid + 512 * r;
        const long long k = wide ? (long long)(((unsigned long long)(unsigned)idx_hi[r] << 32) | (unsigned)idx_lo[r]) : (long long)idx_lo[r];
        const bool ok = i < n_keys && k >= 0 && k < p.Skv;
        if (i < list_tiles * kTK) keys[i] = ok ? (int)k : -1;
        if (ok) mine = i;
        const unsigned long long okm = __ballot(ok);        // a tile is the 32 consecutive entries of half a wavefront
        if ((lane & 31) == 0 && i < list_tiles * kTK) tvalid[i / kTK] = (unsigned)(okm >> (lane & 32)) == 0xffffffffu;
      }
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) mine = max(mine, __shfl_xor(mine, off, 64));
    if (lane == 0) last_valid[wave] = mine;
  };
  // causal padding puts the skipped (-1) slots at the end of a list: tiles past the last valid key do nothing
  auto find_last = [&]() {
    int m = -1;
#pragma unroll
    for (int w = 0; w < 8; ++w) m = max(m, last_valid[w]);
    return __builtin_amdgcn_readfirstlane(m);
  };
  const size_t part_block = (size_t)(((long long)bs * p.G + g) * chunks + chunk) * p.num_splits + split;
  const size_t part_blocks_total = (size_t)p.B * p.S * p.G * chunks * p.num_splits;

  if (producer) {
    // =====================================================================================
    const int sj = role >> 1, hq = role & 1, n = lane & 15, kq = lane >> 4;
    typedef __attribute__((ext_vector_type(4))) unsigned u4;
    // the chunk's query rows as they lie in memory, a quarter of them per producer, then operand order by way of the ring
    constexpr int kQPieces = kDqk / 8;              // 72 pieces of 16 bytes per head row
    constexpr int kQRows = 8 * HB;                  // rows of a producer
    constexpr int kQLoads = kQRows * kQPieces / 64; // 9 HB
    constexpr int kCodePieces = kDqk / 16;          // Q_E8: 36 pieces of 16 codes, two of them to a scale
    constexpr int kCodeLoads = (kQRows * kCodePieces + 63) / 64;
    u4 qload[Q_E8 ? kCodeLoads : kQLoads];
    unsigned char qsc[kCodeLoads];
    if constexpr (Q_E8) {
#pragma unroll
      for (int t = 0; t < kCodeLoads; ++t) {
        const int P = min(lane + 64 * t, kQRows * kCodePieces - 1), hl = P / kCodePieces, piece = P - hl * kCodePieces, h = kQRows * role + hl;
        const size_t row = bs * p.H + head0 + (h < heads_here ? h : 0);
        qload[t] = *reinterpret_cast<const u4*>((const unsigned char*)p.q + row * kDqk + 16 * piece);
        qsc[t] = ((const unsigned char*)p.q_scale)[row * (kDqk / 32) + (piece >> 1)];
      }
    } else
#pragma unroll
    for (int t = 0; t < kQLoads; ++t) {
      const int P = lane + 64 * t, hl = P / kQPieces, piece = P - hl * kQPieces, h = kQRows * role + hl;
      // heads past the end of the group repeat head 0: their columns stay finite and are never stored
      qload[t] = *reinterpret_cast<const u4*>((const unsigned short*)p.q + (bs * p.H + head0 + (h < heads_here ? h : 0)) * (size_t)kDqk + 8 * piece);
    }
    __builtin_amdgcn_sched_barrier(0);
    stage_keys();
    unsigned char* qstage = smem + kLatSlot;        // (no tile is here before the first barrier of the pipeline)
    if constexpr (Q_E8) {
#pragma unroll
      for (int t = 0; t < kCodeLoads; ++t) {
        const int P = min(lane + 64 * t, kQRows * kCodePieces - 1), hl = P / kCodePieces, piece = P - hl * kCodePieces;
        uint4 lo, hi;
        dequant16<false>(make_uint4(qload[t][0], qload[t][1], qload[t][2], qload[t][3]), e8m0_to_f32(qsc[t]), lo, hi);
        *reinterpret_cast<uint4*>(qstage + (kQRows * role + hl) * kQPitch + piece * 32) = lo;
        *reinterpret_cast<uint4*>(qstage + (kQRows * role + hl) * kQPitch + piece * 32 + 16) = hi;
      }
    } else
#pragma unroll
    for (int t = 0; t < kQLoads; ++t) {
      const int P = lane + 64 * t, hl = P / kQPieces, piece = P - hl * kQPieces;
      *reinterpret_cast<u4*>(qstage + (kQRows * role + hl) * kQPitch + piece * 16) = qload[t];
    }
    __syncthreads();                                // keys and query rows are complete
    const int n_tiles = (find_last() + kTK) / kTK;
    bf16x8 qf[HB][18];
#pragma unroll
    for (int gr = 0; gr < HB; ++gr)
#pragma unroll
      for (int ks = 0; ks < 18; ++ks)
        qf[gr][ks] = *reinterpret_cast<const bf16x8*>(qstage + (16 * HB * hq + 16 * gr + n) * kQPitch + (4 * ks + kq) * 16);
    float m_run[HB], l_run[HB];
#pragma unroll
    for (int gr = 0; gr < HB; ++gr) {
      m_run[gr] = -INFINITY;                        // base-2 running reference of head n of the group
      l_run[gr] = 0.0f;                             // this lane's share of its denominator
    }
    // operand reads: row 16 sj + n, piece 4 ks + kq: four lane bases per 256 bytes of the row
    int k_base[4], r_base[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) k_base[i] = (16 * sj + n) * kLatRow + ((4 * i + kq) ^ fold(n)) * 16;
#pragma unroll
    for (int i = 0; i < 2; ++i) r_base[i] = kRopeOff + (16 * sj + n) * kRopeRow + ((4 * i + kq) ^ fold_rope(n)) * 16;
    const int head_l = 16 * HB * hq + n;            // this lane's head of group 0
    // P in the B-operand layout of the 32x32x16 product: lane (head of a 32-head block, key / 8) owns 8 keys
    unsigned char* p_dst = smem + kPOff + (sj * 2 + (HB == 2 ? hq : 0)) * 1024 + ((HB == 2 ? 0 : 16 * hq) + n + (kq >> 1) * 32) * 16 + (kq & 1) * 8;

    __syncthreads();                                // [X] tile 0 has landed
    unsigned lat_off = 0, rope_off = 0;             // of the tile being produced
    for (int t = -1; t < n_tiles; ++t) {
      const int tau = t + 1;
      const bool active = tau < n_tiles;
      f32x4 st[HB];
      if (active) {
        const unsigned char* lat = smem + lat_off;
        const unsigned char* rope = smem + rope_off;
#pragma unroll
        for (int gr = 0; gr < HB; ++gr) st[gr] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 18; ++ks) {
          const bf16x8 k = ks < 16 ? *reinterpret_cast<const bf16x8*>(lat + k_base[ks & 3] + (ks >> 2) * 256)
                                   : *reinterpret_cast<const bf16x8*>(rope + r_base[ks & 1]);
#pragma unroll
          for (int gr = 0; gr < HB; ++gr) mfma_s<F16>(st[gr], k, qf[gr][ks]);
        }
        // this lane: head n of each group, keys 4 kq + i of the sub-tile
        const bool all_valid = tvalid[tau] != 0;    // (uniform)
        int4 kk = make_int4(0, 0, 0, 0);
        if (!all_valid) kk = *reinterpret_cast<const int4*>(keys + tau * kTK + 16 * sj + 4 * kq);
#pragma unroll
        for (int gr = 0; gr < HB; ++gr) {
#pragma unroll
          for (int i = 0; i < 4; ++i) st[gr][i] *= qk_scale;
          if (!all_valid) {
            st[gr][0] = kk.x >= 0 ? st[gr][0] : -INFINITY;
            st[gr][1] = kk.y >= 0 ? st[gr][1] : -INFINITY;
            st[gr][2] = kk.z >= 0 ? st[gr][2] : -INFINITY;
            st[gr][3] = kk.w >= 0 ? st[gr][3] : -INFINITY;
          }
          const float mx = max_rows(vmax(vmax3(st[gr][0], st[gr][1], st[gr][2]), st[gr][3]));
          if (lane < 16) maxbuf[sj * 64 + head_l + 16 * gr] = mx;
        }
      }
      __syncthreads();                              // [M] both sub-tiles' maxima are there
      if (active) {
        const int par = tau & 1;
        float mx[HB];
        bool grow = false, rescale = false;
#pragma unroll
        for (int gr = 0; gr < HB; ++gr) {
          mx[gr] = vmax(maxbuf[head_l + 16 * gr], maxbuf[64 + head_l + 16 * gr]);
          const bool up = mx[gr] > m_run[gr] + kLazy;
          grow |= up;
          // accumulators of a head whose reference was -inf are still zero: nothing to rescale
          rescale |= up && m_run[gr] != -INFINITY;
        }
        const bool any_rescale = __ballot(rescale) != 0ull;
        if (lane == 0 && sj == 0) flagbuf[par * 2 + hq] = any_rescale;
        if (__ballot(grow) != 0ull) {               // (both producers of the heads decide alike)
#pragma unroll
          for (int gr = 0; gr < HB; ++gr) {
            float fac = 1.0f;
            if (mx[gr] > m_run[gr] + kLazy) {
              fac = m_run[gr] == -INFINITY ? 1.0f : fast_exp2(m_run[gr] - mx[gr]);
              l_run[gr] *= fac;
              m_run[gr] = mx[gr];
            }
            if (any_rescale && sj == 0 && lane < 16) facbuf[par * 64 + head_l + 16 * gr] = fac;
          }
        }
#pragma unroll
        for (int gr = 0; gr < HB; ++gr) {
          // exp2(-inf - m) is 0 for a finite m; a head with no valid key yet keeps m_run = -inf
          const float m = vmax(m_run[gr], -1.0e30f);
          float pr[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pr[i] = fast_exp2(st[gr][i] - m);
            l_run[gr] += pr[i];
          }
          *reinterpret_cast<uint2*>(p_dst + par * 4096 + gr * 256) =
              F16 ? make_uint2(pack_f16(pr[0], pr[1]), pack_f16(pr[2], pr[3])) : make_uint2(pack_bf16(pr[0], pr[1]), pack_bf16(pr[2], pr[3]));
        }
      }
      lat_off = lat_off + kLatSlot == kRing * kLatSlot ? 0u : lat_off + kLatSlot;
      rope_off = rope_off + kRopeSlot == kRopeRing * kRopeSlot ? 0u : rope_off + kRopeSlot;
      __syncthreads();                              // [E_t]
    }
#pragma unroll
    for (int gr = 0; gr < HB; ++gr) {
      l_run[gr] += xor16(l_run[gr]);
      l_run[gr] += xor32(l_run[gr]);
      if (lane < 16) {
        stats[(sj * 64 + head_l + 16 * gr) * 2 + 0] = m_run[gr];
        stats[(sj * 64 + head_l + 16 * gr) * 2 + 1] = l_run[gr];
      }
    }
    __syncthreads();                                // [S] statistics are visible; the ring is free
    return;
  }

  // =======================================================================================
  // consumer c = role: value channels 128c .. 128c+127 of every head; also the row loads
  // =======================================================================================
  stage_keys();
  __syncthreads();                                  // keys[] is complete
  const int last = find_last();
  const int n_tiles = (last + kTK) / kTK;
  const int spare_row = n_tiles > 0 ? __builtin_amdgcn_readfirstlane(keys[max(last, 0)]) : 0;
  // HBM -> LDS.  A skipped key fetches the list's last valid row instead (its probability is zero), so every tile is
  // the same nine load instructions per wavefront and the in-order load counter can be waited on by count.  The loads
  // are inline assembly (the compiler would otherwise order every later LDS read behind them) with a uniform 64-bit
  // base and a 32-bit byte offset per lane: rows 8c .. 8c+7, one instruction each, and their rope tails, one for all.
  const size_t group_row0 = ((size_t)b * p.Skv_pitch) * p.G + g;     // cache row of key 0; key k is G rows further per step
  const bool packed = p.d_kv == kDqk;
  const unsigned row_bytes = (unsigned)p.d_kv * 2u;
  const unsigned char* lat_base = (const unsigned char*)p.kv + group_row0 * row_bytes;
  const unsigned char* rope_base = packed ? lat_base + kLatRow : (const unsigned char*)p.rope + group_row0 * kRopeRow;
  const unsigned lat_step = (unsigned)p.G * row_bytes, rope_step = packed ? lat_step : (unsigned)p.G * kRopeRow;
  const unsigned smem_base = (unsigned)(size_t)(lds_void*)smem;
  auto dma16 = [&](const unsigned char* base, unsigned off, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
  };
  unsigned dma_lat = 0, dma_rope = 0, row_off = 0, tail_off = 0;
  const unsigned tail_lane = (unsigned)((lane & 7) ^ fold_rope((8 * role + (lane >> 3)) & 15)) * 16u;
  auto dma_prepare = [&](int tau, unsigned lat_slot, unsigned rope_slot) {
    dma_lat = smem_base + lat_slot + (unsigned)role * 8u * kLatRow;
    dma_rope = smem_base + kRopeOff + rope_slot + (unsigned)role * 8u * kRopeRow;
    const int* tk = keys + tau * kTK + 8 * role;
    const int k = tk[lane & 7], kt = tk[lane >> 3];
    row_off = (unsigned)(k >= 0 ? k : spare_row) * lat_step;        // of row lane % 8
    tail_off = (unsigned)(kt >= 0 ? kt : spare_row) * rope_step + tail_lane;
  };
  auto dma_part = [&](int i) {                      // i a constant
    if (i < 8) {
      const unsigned row = __builtin_amdgcn_readlane(row_off, i);
      // (rows 8c + i: row within 16 is 8 (c % 2) + i)
      const unsigned f = (role & 1) ? (unsigned)fold(8 + i) : (unsigned)fold(i);
      dma16(lat_base, row + (((unsigned)lane ^ f) << 4), dma_lat + i * kLatRow);
    } else {
      dma16(rope_base, tail_off, dma_rope);
    }
  };

  // ---- value side state: o[dvb][hb] = O^T[32 channels x 32 heads] ----
  f32x16 o[4][HB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int hb = 0; hb < HB; ++hb)
#pragma unroll
      for (int j = 0; j < 16; ++j) o[i][hb][j] = 0.0f;
  // transposing reads of V^T: a 16-lane group covers columns 16 (group % 2) .. of a 32-channel block and rows
  // 8 (lane / 32) + 0..3 (first read) and + 4..7 (second); lane i of it supplies row i / 4, columns 4 (i % 4) ..
  int v_base[2][4];
  {
    const int i16 = lane & 15, cc = 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1), r0 = 8 * (lane >> 5) + (i16 >> 2);
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int dvb = 0; dvb < 4; ++dvb)
        v_base[half][dvb] = (r0 + 4 * half) * kLatRow + role * 256 + (((4 * dvb + cc) ^ fold(r0 + 4 * half)) << 4) + (i16 & 1) * 8;
  }
  auto tr16 = [&](int at) {
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + at)));
  };
  const unsigned char* p_lane = smem + kPOff + lane * 16;
  // one 16-key step of the value product of the tile in the slot at `slot`; the loads of the tile to fetch go between
  // the products (issuing blocks while the load unit's queue is full)
  auto value_step = [&](int par, int kstep, unsigned slot, bool dma) {
    bf16x8 pb[HB];
#pragma unroll
    for (int hb = 0; hb < HB; ++hb) pb[hb] = *reinterpret_cast<const bf16x8*>(p_lane + par * 4096 + (kstep * 2 + hb) * 1024);
    bf16x8 a[4];
#pragma unroll
    for (int dvb = 0; dvb < 4; ++dvb) {
      const bf16x4 a0 = tr16((int)slot + v_base[0][dvb] + kstep * 16 * kLatRow), a1 = tr16((int)slot + v_base[1][dvb] + kstep * 16 * kLatRow);
      a[dvb][0] = a0[0]; a[dvb][1] = a0[1]; a[dvb][2] = a0[2]; a[dvb][3] = a0[3];
      a[dvb][4] = a1[0]; a[dvb][5] = a1[1]; a[dvb][6] = a1[2]; a[dvb][7] = a1[3];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int dvb = 0; dvb < 4; ++dvb) {
#pragma unroll
      for (int hb = 0; hb < HB; ++hb) mfma_o<F16>(o[dvb][hb], a[dvb], pb[hb]);
      if (dma) {
        dma_part(kstep * 4 + dvb);
        if (kstep == 1 && dvb == 3) dma_part(8);
      }
    }
  };

  // ---- pipeline ----
  if (n_tiles > 0) {
    dma_prepare(0, 0u, 0u);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) dma_part(i);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();                                  // [X] tile 0 has landed
#pragma unroll
  for (int tau = 1; tau < kAhead; ++tau)
    if (tau < n_tiles) {
      dma_prepare(tau, (unsigned)tau * kLatSlot, (unsigned)tau * kRopeSlot);
#pragma unroll
      for (int i = 0; i < kLoads; ++i) dma_part(i);
    }
  __syncthreads();                                  // [M_-1]
  if (n_tiles > 2) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();                                  // [E_-1] tile 1 has landed
  unsigned cur = 0, fetch_lat = 3 * kLatSlot, fetch_rope = 0;      // slots of tile t and of tile t + 3
  for (int t = 0; t < n_tiles; ++t) {
    const bool dma = t + kAhead < n_tiles;
    const int par = t & 1;
    if (dma) dma_prepare(t + kAhead, fetch_lat, fetch_rope);
    if (__builtin_amdgcn_readfirstlane(flagbuf[par * 2] | flagbuf[par * 2 + 1]) != 0) {      // producers moved a reference: rescale (rare)
      const int hd = lane & 31;
#pragma unroll
      for (int hb = 0; hb < HB; ++hb) {
        const int h = 32 * hb + hd;
        const float fsc = flagbuf[par * 2 + h / (16 * HB)] ? facbuf[par * 64 + h] : 1.0f;
#pragma unroll
        for (int dvb = 0; dvb < 4; ++dvb)
#pragma unroll
          for (int j = 0; j < 16; ++j) o[dvb][hb][j] *= fsc;
      }
    }
    value_step(par, 0, cur, dma);
    __syncthreads();                                // [M_t]
    value_step(par, 1, cur, dma);
    // tile t + 2 must have landed before the next barrier; the tile just issued may stay in flight
    if (dma) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    cur = cur + kLatSlot == kRing * kLatSlot ? 0u : cur + kLatSlot;
    fetch_lat = fetch_lat + kLatSlot == kRing * kLatSlot ? 0u : fetch_lat + kLatSlot;
    fetch_rope = fetch_rope + kRopeSlot == kRopeRing * kRopeSlot ? 0u : fetch_rope + kRopeSlot;
    __syncthreads();                                // [E_t]
  }
  __syncthreads();                                  // [S] statistics are visible; the ring is free

  // ---- epilogue ----
  const int hd = lane & 31, gq2 = lane >> 5;
  float* xbuf = reinterpret_cast<float*>(smem) + role * 32 * kXPitch;     // private to this wavefront
#pragma unroll
  for (int hb = 0; hb < HB; ++hb) {
    const int h_local = 32 * hb + hd;
    const float m_all = stats[h_local * 2], l_all = stats[h_local * 2 + 1] + stats[(64 + h_local) * 2 + 1];
    if (p.num_splits != 1) {
      // key split: the unnormalised accumulators leave as the lanes hold them: [consumer][head block][dvb][row pair][lane][8]
      float* blk = (float*)p.workspace + part_block * (size_t)(HB * kMlaPartFloats) + ((size_t)((role * HB + hb) * 8) * 64 + lane) * 8;
#pragma unroll
      for (int dvb = 0; dvb < 4; ++dvb)
#pragma unroll
        for (int j4 = 0; j4 < 4; ++j4) {
          const f32x16& acc = o[dvb][hb];
          *reinterpret_cast<float4*>(blk + (size_t)(dvb * 2 + (j4 >> 1)) * 512 + (j4 & 1) * 4) =
              make_float4(acc[4 * j4], acc[4 * j4 + 1], acc[4 * j4 + 2], acc[4 * j4 + 3]);
        }
      if (role == 0 && lane < 32) {
        float* ml = (float*)p.workspace + part_blocks_total * (size_t)(HB * kMlaPartFloats) + (part_block * kHeadsWg + h_local) * 2;
        ml[0] = m_all;
        ml[1] = l_all;
      }
      continue;
    }
    float out_scale = 1.0f, lse_val = 0.0f;
    {
      float m_fin = m_all, l_fin = l_all;
      if (mla_has_sinks(p) && h_local < heads_here) {
        const float sk = p.sinks[head0 + h_local] * kLog2e;
        const float m2 = fmaxf(m_fin, sk);
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
    // transpose through LDS: lane (head hd, gq2) holds channels 32dvb + 8j + 4gq2 + (0..3) in o[.][4j..4j+3]
#pragma unroll
    for (int dvb = 0; dvb < 4; ++dvb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x16& acc = o[dvb][hb];
        *reinterpret_cast<float4*>(xbuf + hd * kXPitch + 32 * dvb + 8 * j + 4 * gq2) =
            make_float4(acc[4 * j] * out_scale, acc[4 * j + 1] * out_scale, acc[4 * j + 2] * out_scale, acc[4 * j + 3] * out_scale);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // rows of 128 channels leave coalesced: 16 lanes x 8 channels, four heads per step
#pragma unroll 4
    for (int it = 0; it < 8; ++it) {
      const int row = 4 * it + (lane >> 4), c8 = (lane & 15) * 8;
      const int hl = 32 * hb + row;
      if (hl >= heads_here) continue;
      const float4 v = *reinterpret_cast<const float4*>(xbuf + row * kXPitch + c8);
      const float4 u = *reinterpret_cast<const float4*>(xbuf + row * kXPitch + c8 + 4);
      const size_t off = (bs * p.H + head0 + hl) * (size_t)kLat + 128 * role + c8;
      if (p.out_dtype == CPPMEGA_MI355_F32) {
        *reinterpret_cast<float4*>((float*)p.out + off) = v;
        *reinterpret_cast<float4*>((float*)p.out + off + 4) = u;
      } else if (p.out_dtype == CPPMEGA_MI355_BF16) {
        *reinterpret_cast<uint4*>((unsigned short*)p.out + off) =
            make_uint4(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w), pack_bf16(u.x, u.y), pack_bf16(u.z, u.w));
      } else {
        *reinterpret_cast<uint4*>((unsigned short*)p.out + off) =
            make_uint4(pack_f16(v.x, v.y), pack_f16(v.z, v.w), pack_f16(u.x, u.y), pack_f16(u.z, u.w));
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (role == 0 && lane < 32 && h_local < heads_here && p.lse) p.lse[bs * p.H + head0 + h_local] = lse_val;
  }
}

// Rows of 576 e4m3 codes and 18 E8M0 bytes as bf16, 16 codes per thread: the cache, [B, Skv, G, 576], then, for the kernel of 16
// heads, the queries behind it (q_out), [B, S, H, 576].
__global__ __launch_bounds__(256) void sparse_mla_e8m0_rows_kernel(const MlaParams p, unsigned short* out, unsigned short* q_out) {
  constexpr unsigned kPieces = kDqk / 16;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t row = i / kPieces, cache_rows = (size_t)p.B * p.Skv * p.G;
  const unsigned piece = (unsigned)(i - row * kPieces);
  const bool of_q = row >= cache_rows;
  if (of_q && (!q_out || row - cache_rows >= (size_t)p.B * p.S * p.H)) return;
  const size_t per_batch = (size_t)p.Skv * p.G, b = row / per_batch;
  const size_t src = of_q ? row - cache_rows : b * ((size_t)p.Skv_pitch * p.G) + (row - b * per_batch);
  uint4 lo, hi;
  dequant16<false>(*reinterpret_cast<const uint4*>((const unsigned char*)(of_q ? p.q : p.kv) + src * kDqk + 16 * piece),
                   e8m0_to_f32(((const unsigned char*)(of_q ? p.q_scale : p.kv_scale))[src * (kDqk / 32) + (piece >> 1)]), lo, hi);
  uint4* dst = reinterpret_cast<uint4*>((of_q ? q_out : out) + (of_q ? src : row) * kDqk + 16 * piece);
  dst[0] = lo;
  dst[1] = hi;
}

bool e8m0_rows(const MlaParams& p) {
  return p.q_dtype == CPPMEGA_MI355_E4M3 && p.kv_dtype == CPPMEGA_MI355_E4M3 && p.q_scale_kind == CPPMEGA_MI355_SCALE_E8M0 &&
         p.kv_scale_kind == CPPMEGA_MI355_SCALE_E8M0 && p.q_scale_block == 32 && p.kv_scale_block == 32 && p.q_scale && p.kv_scale;
}
size_t e8m0_row_bytes(const MlaParams& p) { return e8m0_rows(p) ? ((size_t)p.B * p.Skv * p.G * kDqk * 2 + 255) & ~(size_t)255 : 0; }

bool rows_of_16_bits(const MlaParams& p) {
  if (e8m0_rows(p)) {
    // Every row of the cache is converted, for 1152 bytes of workspace and 0.35 ns each.  Up to 65536 rows (25 us) that is
    // made up for by short lists too (8 x 256 of 65536: 43 / 48 / 47 us with 16 / 64 / 128 heads, 41 / 68 / 70 on the tile
    // kernel); beyond, where the lists name two keys for every row (2 M keys of 1 M rows: 715 / 796 / 1058 us against 698 /
    // 1159 / 1189; 1 M keys: 538 / 571 / 690 against 363 / 583 / 594).  And never for more than the scratch kept between calls.
    const long long rows = (long long)p.B * p.Skv * p.G;
    return p.plan_level == 0 && p.d_kv == kDqk && p.rope_dim == 0 &&
           (rows <= 65536 || (2 * rows <= (long long)p.B * p.S * p.G * p.topk && e8m0_row_bytes(p) <= ((size_t)1 << 30)));
  }
  if ((p.q_dtype != CPPMEGA_MI355_BF16 && p.q_dtype != CPPMEGA_MI355_F16) || p.kv_dtype != p.q_dtype) return false;
  if (p.q_scale_kind != CPPMEGA_MI355_SCALE_NONE || p.kv_scale_kind != CPPMEGA_MI355_SCALE_NONE) return false;
  return true;
}

}  // namespace

bool sparse_mla_rows16_supported(const MlaParams& p) {
  if (!rows_of_16_bits(p)) return false;
  if (p.d_qk != kDqk || p.d_v != kLat || p.d_kv + p.rope_dim != kDqk) return false;
  if (p.rope_dim != 0 && (p.rope_dim != kRope || p.rope_dtype != p.q_dtype)) return false;
  if (p.topk < 1 || (size_t)p.B * p.S == 0) return false;
  if (((uintptr_t)p.q | (uintptr_t)p.kv | (uintptr_t)p.rope) & 15) return false;
  // a lane's byte offset from the first row of its batch, and cache rows, are counted in 32 bits
  if ((unsigned long long)p.Skv_pitch * p.G * kDqk * 2 >= (1ull << 32) || (unsigned long long)p.B * p.Skv_pitch * p.G >= 0x7fffffffull) return false;
  return p.topk <= 16 * kMaxKeys;                 // the combine step merges at most 16 key splits
}

size_t sparse_mla_e8m0_copy_bytes(const MlaParams& p) {
  return e8m0_rows(p) ? e8m0_row_bytes(p) + (((size_t)p.B * p.S * p.H * kDqk * 2 + 255) & ~(size_t)255) : 0;
}

int sparse_mla_e8m0_copy(MlaParams& p, hipStream_t stream) {
  const size_t cache = e8m0_row_bytes(p), all = sparse_mla_e8m0_copy_bytes(p);
  const size_t pieces = ((size_t)p.B * p.Skv * p.G + (size_t)p.B * p.S * p.H) * (kDqk / 16);
  unsigned short *rows = (unsigned short*)p.workspace, *q = (unsigned short*)((char*)p.workspace + cache);
  hipLaunchKernelGGL(sparse_mla_e8m0_rows_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, p, rows, q);
  CM_HIP_CHECK(hipGetLastError());
  p.kv = rows;
  p.q = q;
  p.Skv_pitch = p.Skv;
  p.workspace = (char*)p.workspace + all;
  p.q_dtype = p.kv_dtype = CPPMEGA_MI355_BF16;
  p.q_scale_kind = p.kv_scale_kind = CPPMEGA_MI355_SCALE_NONE;
  return 0;
}

double sparse_mla_rows16_plan(MlaParams& p) {
  p.rows16 = 1;
  p.heads_per_wg = p.heads_per_group <= 32 ? 32 : 64;
  const int chunks = (p.heads_per_group + p.heads_per_wg - 1) / p.heads_per_wg;
  const long long base = (long long)p.B * p.S * p.G * chunks;
  return mla_key_splits(p, base, kMaxKeys, p.heads_per_wg == 64 ? 1.1 : 0.85, p.heads_per_wg, false);
}

int sparse_mla_rows16_launch(const MlaParams& args, hipStream_t stream) {
  MlaParams p = args;
  const int chunks = (p.heads_per_group + p.heads_per_wg - 1) / p.heads_per_wg;
  const long long wgs = (long long)p.B * p.S * p.G * p.num_splits * chunks;
  if (wgs > 0x7fffffffll || p.keys_per_split > kMaxKeys || p.num_splits > 16)
    return fail(CPPMEGA_MI355_ERR_UNSUPPORTED, "sparse MLA: launch too large");
  const bool f16 = p.q_dtype == CPPMEGA_MI355_F16, e8 = e8m0_rows(p);
  if (e8) {
    const size_t pieces = (size_t)p.B * p.Skv * p.G * (kDqk / 16);
    hipLaunchKernelGGL(sparse_mla_e8m0_rows_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, args, (unsigned short*)args.workspace, (unsigned short*)nullptr);
    CM_HIP_CHECK(hipGetLastError());
    p.kv = args.workspace;
    p.Skv_pitch = p.Skv;
    p.workspace = (char*)args.workspace + e8m0_row_bytes(args);
  }
  void (*kernel)(MlaParams) = e8 ? (p.heads_per_wg == 64 ? sparse_mla_rows16_kernel<false, 2, true> : sparse_mla_rows16_kernel<false, 1, true>)
                            : p.heads_per_wg == 64 ? (f16 ? sparse_mla_rows16_kernel<true, 2> : sparse_mla_rows16_kernel<false, 2>)
                                                   : (f16 ? sparse_mla_rows16_kernel<true, 1> : sparse_mla_rows16_kernel<false, 1>);
  CM_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kSmem));
  hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(512), kSmem, stream, p);
  CM_HIP_CHECK(hipGetLastError());
  return p.num_splits > 1 ? sparse_mla_combine_f32(p, stream) : 0;
}

size_t sparse_mla_rows16_workspace_bytes(const MlaParams& p) {
  if (p.num_splits <= 1) return e8m0_row_bytes(p);
  const int chunks = (p.heads_per_group + p.heads_per_wg - 1) / p.heads_per_wg;
  const size_t blocks = (size_t)p.B * p.S * p.G * chunks * p.num_splits;
  return e8m0_row_bytes(p) + blocks * (size_t)(p.heads_per_wg / 32 * kMlaPartFloats + p.heads_per_wg * 2) * sizeof(float);
}

}  // namespace cm
