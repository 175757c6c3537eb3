// FP8 (e4m3) block-scaled weight GEMM for batches and prefill chunks (gfx950).
//
//   out[m, n] = sum_k dec(w[n, k]) * w_scale(n, k / 128) * x[m, k],   x bf16 or fp16, fp32 accumulation
//
// The kernels of fp8_vecmat.hip read the whole weight once per 4 to 16 activation rows; from 17 rows on a
// tile of both operands is worth staging in LDS.  The load unit writes the tiles there itself (global_load_lds, pieces of
// 128 bytes of a row: such loads reach 50 B/clk a CU, pieces of 64 bytes 28, of 16 bytes 10), as many stages ahead as the
// LDS holds.  Measured (microseconds a call in a row of calls over three weights in turn, bf16 results; through registers, two stages
// ahead -> here), M x N x K, scales per 128 x 128 / per row and 128 channels:
//   2048 x 8192 x 1536  64 -> 59 / 65 -> 60            2048 x 7168 x 16384  466 -> 444 = 1080 TFLOP/s / 535 -> 474
//   1040 x 2621 x 5248  54 -> 41 / 58 -> 43            879 x 1007 x 6528    45 -> 23 / 48 -> 25
//   231 x 4895 x 10240  52 -> 36 / 56 -> 40            32 x 7168 x 16384    29.1 -> 25.6 / 35.2 -> 33.0
//   55 x 2804 x 640     7.9 -> 6.1 / 7.9 -> 6.3
// (Under the profiler, whose calls do not overlap, 32 x 7168 x 16384 with a scale per row is 33 us and 4.6 for the sum of the splits, as before.)
// What bounds it: a large product, no unit alone: of 5070 clocks a 128 x 256 x 128 stage with its share of a tile's ends (2048 x 8192 x 1536) 2048
// are products on each SIMD, 1630 other vector instructions, 1770 the LDS (operand reads and, at 128 B/clk, arriving rows), and two
// wavefronts cover each other's phases in part; a small one, launch, first loads and stores (5 us); a small batch, the weights' stream.

#include <stdint.h>

#include "fp8_vecmat.h"
#include "mfma_util.h"

namespace cm {
namespace {

// 8 e4m3 codes -> the bf16 / fp16 values they stand for (exact)
template <bool F16>
__device__ __forceinline__ u32x4 codes8(unsigned a, unsigned b) {
  u32x4 r;
  if (F16) {
    r[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 1.0f, false));
    r[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 1.0f, true));
    r[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 1.0f, false));
    r[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 1.0f, true));
  } else {
    r[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.0f, false));
    r[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.0f, true));
    r[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.0f, false));
    r[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.0f, true));
  }
  return r;
}

template <bool F16>
__device__ __forceinline__ f32x4 product(const u32x4& a, const u32x4& b, const f32x4& c) {
  return mm<F16>(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c);
}

// floats from one split's sums to the next: whole 16-byte pieces
__host__ __device__ __forceinline__ size_t split_step(int m, int n) { return ((size_t)m * n + 3) & ~(size_t)3; }

// Which of the eight 16-byte places of its 128-byte LDS row a piece lies in: piece ^ fold(row).  A 16-byte read is
// served sixteen lanes (all banks) at a time: sixteen rows with one piece, or with the pieces of neighbouring quarters
// of the wavefront; either way the pairs of rows fall on eight different places.
__device__ __forceinline__ int fold(int row) { return ((((row >> 3) ^ (row >> 2)) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 1) & 1); }

// A workgroup's tile: WM x WN wavefronts of TM x TN tiles of 16 x 16, and WK such groups, which take the 128-channel blocks
// in turn (two groups add their sums in LDS at the end: half the steps of a tile where the tiles leave CUs idle, without a
// second launch).  A stage is a block per group: [group][half block][row][128 bytes] of activations, [group][row][128 bytes]
// of weights and every wavefront's weight scales.  PERSIST: a workgroup goes on to its next tile, whose first stages are on
// their way under the last products and the stores of the one before.
template <int TM_, int TN_, int WM_, int WN_, int WK_, int SLOTS_, bool PERSIST_>
struct Tile {
  static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, WK = WK_, SLOTS = SLOTS_;
  static constexpr bool PERSIST = PERSIST_;
  static constexpr int kWaves = WM * WN * WK, kThreads = 64 * kWaves;
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  static constexpr int XL = WK * 2 * BM / 8 / kWaves, WL = WK * BN / 8 / kWaves;    // load instructions per wavefront and stage
  static_assert(XL * kWaves * 8 == WK * 2 * BM && WL * kWaves * 8 == WK * BN, "whole instructions per wavefront");
  static constexpr int kX = WK * 2 * BM * 128, kW = WK * BN * 128, kS = kWaves * 256;
  static constexpr int kStage = kX + kW + kS;                                        // bytes of one slot
  static constexpr int PITCH = TN * 16 + 4;                                          // floats of a row on its way out
  static constexpr int kOut = kWaves * 16 * PITCH * 4;
  static constexpr int kLds = SLOTS * kStage + (PERSIST ? kOut : 0);
  static_assert(WK == 1 || (WK == 2 && !PERSIST), "the sums of two groups meet in the stages' place");
};

// Every 128-channel block is accumulated from zero and enters the sums as acc += scale * tile, so fp32
// scales of any kind are applied exactly; in the product layout (weights as the second operand) a lane
// holds one output channel, i.e. one scale per tile.  A lane's 16 weight bytes feed two products: the
// contraction runs over the channels in the order the bytes lie in, and the activation pieces follow it.
//
// SECTIONS, for float32 results: the error of a sum grows with the number of blocks that are added one after the other, so from six on
// about sqrt(n) sections of blocks are added up by themselves and then to a second sum.  Without it the plans of few splits lost
// digits: rms error against float64, one chain / here, 790 x 9331 x 7168 1.37e-7 / 0.80e-7 (two splits of 28 blocks 1.03e-7), 676 x 2255
// x 6656 1.00e-7 / 0.74e-7 (four splits 0.82e-7).  It costs up to 3 % of a call, and results of 16 bits do not show it.
template <class T, bool F16, bool SECTIONS>
__global__ __launch_bounds__(T::kThreads, 2) void fp8_gemm_kernel(const VecmatParams p) {
  constexpr int TM = T::TM, TN = T::TN, WM = T::WM, WN = T::WN, WK = T::WK, SLOTS = T::SLOTS, BM = T::BM, BN = T::BN, XL = T::XL, WL = T::WL;
  constexpr int PITCH = T::PITCH, L = XL + WL + 1;
  __shared__ u32x4 smem[T::kLds / 16];
  char* const lds = reinterpret_cast<char*>(smem);

  const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (WM * WN), wm = (wave / WN % WM) * TM * 16, wn = (wave % WN) * TN * 16;
  const int quad = lane >> 4, l16 = lane & 15;

  const int tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  const int blocks = p.k / 128;
  const int b0 = (int)((long long)blocks * blockIdx.y / p.k_splits), b1 = (int)((long long)blocks * (blockIdx.y + 1) / p.k_splits);
  const int stages = (b1 - b0 + WK - 1) / WK;
  int turned = 0;                                                    // the stage it begins with (two groups)
  // Stages come in sections of `section` or, the last `longer` ones, one more.
  const int sections = SECTIONS && stages > 5 ? __builtin_amdgcn_readfirstlane((int)__builtin_amdgcn_sqrtf((float)stages - 1.5f)) : 1;
  const int section = stages / sections, longer = stages - section * sections;

  // Rows and columns of tile e.  Consecutive workgroups go round the eight XCDs: every XCD takes one run of
  // the order (groups of eight column tiles; inside, row tile by row tile), so that its L2 holds the
  // weights of a group while the row tiles pass.  (The number of workgroups that take several tiles is a multiple of 8.)
  auto place = [&](int e, int& m0, int& n0) {
    const int q = total >> 3, r = total & 7, xcd = e & 7;
    const int t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (e >> 3);
    const int per_group = tiles_m * 8, group = t / per_group;
    const int width = tiles_n - group * 8 < 8 ? tiles_n - group * 8 : 8;
    const int in_group = t - group * per_group;
    m0 = (in_group / width) * BM;
    n0 = (group * 8 + in_group % width) * BN;
  };

  // ---- loads: inline assembly (the compiler would order every later LDS read behind them), waited for by count ----
  // One uniform base per operand, moved on by a stage at a time, and 32-bit lane offsets.  An instruction moves eight rows
  // of 128 bytes.
  const char *xbase, *wbase, *sbase;
  unsigned xoff[XL], woff[WL], soff;
  int next_e = (int)blockIdx.x, next_b = b0, left;                   // tile and block to be requested next; stages not requested
  auto start = [&]() {
    int m0, n0;
    place(next_e, m0, n0);
    // Column tiles begin at different places of K and go round: where rows are a power of two of bytes apart, workgroups in step
    // ask the same memory channels (20 x 7168 x 16384 30.5 -> 25.9 us, as the last step of a decode layer 33 -> 28; 30 x 4096 x 14336
    // 17 -> 15.7).  Only while an XCD's L2 holds the activations, whose tiles are then read at different times: with row
    // tiles that fetched their weights at different times 1388 x 1098 x 9472 took 60 us for 43.
    if (WK == 2 && (size_t)p.m * p.k * 2 <= (2u << 20)) turned = (int)((unsigned)(n0 / BN) * 5u % (unsigned)stages);
    next_b = b0 + turned * WK;
    xbase = reinterpret_cast<const char*>(p.x) + ((size_t)m0 * p.k + (size_t)next_b * 128) * 2;
    wbase = reinterpret_cast<const char*>(p.w) + (size_t)n0 * p.k + (size_t)next_b * 128;
    const int first = n0 >> p.srow_shift;
    sbase = reinterpret_cast<const char*>(p.scale_w) + ((size_t)first * p.srow_stride + (size_t)next_b * p.scol_stride) * 4;
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int u = wave * XL + i, plane = u & 1, rg = (u >> 1) / WK;
      const int row = rg * 8 + (lane >> 3), m = m0 + row < p.m ? row : p.m - 1 - m0;       // rows past the end repeat the last one and are not stored
      xoff[i] = (unsigned)m * (unsigned)p.k * 2u + (unsigned)plane * 128u + 16u * (unsigned)((lane & 7) ^ fold(row));
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int u = wave * WL + i, rg = u / WK;
      const int row = rg * 8 + (lane >> 3), n = n0 + row < p.n ? row : p.n - 1 - n0;
      woff[i] = (unsigned)n * (unsigned)p.k + 16u * (unsigned)((lane & 7) ^ fold(row));
    }
    const int c = n0 + wn + lane % (TN * 16), n = c < p.n ? c : p.n - 1;
    soff = (unsigned)((n >> p.srow_shift) - first) * (unsigned)p.srow_stride * 4u;
  };
  const unsigned lds_base = (unsigned)(size_t)(lds_void*)smem;
  auto load16 = [&](const char* base, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(off), "s"(base) : "memory", "m0");
  };
  // Weights that one row tile reads, of a size that the last-level cache (256 MB) does not keep for the next call beside what else a
  // program runs: non-temporal, so that they push nothing out (20 x 7168 x 16384 25.9 -> 24.4 us, a decode layer of 18 to 32 sequences
  // 3 to 5 us).  Smaller ones may still be there (three takes in turn of 30 x 4096 x 14336 15.7 / 17.7 us, of 24 x 10000 x 2048 9.9 / 11.6).
  const bool once = tiles_m == 1 && (size_t)p.n * p.k >= (64u << 20);
  auto load16_once = [&](const char* base, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(to), "v"(off), "s"(base) : "memory", "m0");
  };
  auto load4 = [&](const char* base, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(to), "v"(off), "s"(base) : "memory", "m0");
  };
  unsigned next_slot = lds_base;
  // requests instruction i of the next stage (of the same number whatever the stage holds: a block that is not there
  // repeats its neighbour)
  auto issue = [&](int i) {
    const bool pair = WK == 1 || next_b + 1 < b1;
    if (i < WL) {
      const int u = wave * WL + i, g = u % WK, rg = u / WK;
      const char* const at = wbase + (pair ? g * 128 : 0);
      const unsigned to = next_slot + (unsigned)(T::kX + (g * BN + rg * 8) * 128);
      if (BM == 32 && once) load16_once(at, woff[i], to);
      else load16(at, woff[i], to);
    } else if (i < XL + WL) {
      const int u = wave * XL + i - WL, plane = u & 1, g = (u >> 1) % WK, rg = (u >> 1) / WK;
      load16(xbase + (pair ? g * 256 : 0), xoff[i - WL], next_slot + (unsigned)(((g * 2 + plane) * BM + rg * 8) * 128));
    } else {
      load4(sbase + (pair ? (size_t)wk * p.scol_stride * 4 : 0), soff, next_slot + (unsigned)(T::kX + T::kW + wave * 256));
      xbase += WK * 256;
      wbase += WK * 128;
      sbase += (size_t)WK * p.scol_stride * 4;
      next_b += WK;
      --left;
      next_slot = next_slot + T::kStage == lds_base + SLOTS * T::kStage ? lds_base : next_slot + T::kStage;
      if (WK == 2 && next_b >= b1) {
        next_b = b0;
        xbase -= (size_t)stages * (WK * 256);
        wbase -= (size_t)stages * (WK * 128);
        sbase -= (size_t)stages * WK * p.scol_stride * 4;
      }
      if (T::PERSIST && next_b >= b1 && left > 0) {
        next_e += (int)gridDim.x;
        start();
      }
    }
  };

  f32x4 acc[TM][TN], tile[TM][TN], sum[SECTIONS ? TM : 1][SECTIONS ? TN : 1];
  const int xlane = (wk * 2 * BM + wm + l16) * 128, wlane = T::kX + (wk * BN + wn + l16) * 128, slane = T::kX + T::kW + wave * 256 + l16 * 4;
  const int f = fold(l16);
  const int xpos[2] = {xlane + 16 * ((quad * 2) ^ f), xlane + 16 * ((quad * 2 + 1) ^ f)};
  const int wpos[2] = {wlane + 16 * (quad ^ f), wlane + 16 * ((4 + quad) ^ f)};
  u32x4 wr[2][TN], xr[2][TM];
  float sc[TN];
  auto read_w = [&](int slot, int c) {
#pragma unroll
    for (int j = 0; j < TN; ++j) wr[c][j] = *reinterpret_cast<const u32x4*>(lds + slot + wpos[c] + j * 2048);
  };
  auto read_x = [&](int slot, int c, int h) {
#pragma unroll
    for (int i = 0; i < TM; ++i) xr[h][i] = *reinterpret_cast<const u32x4*>(lds + slot + xpos[h] + c * BM * 128 + i * 2048);
  };
  // products of channels 64 c + 16 quad + 8 h .. of the block; loads of the stage after next go between their columns
  // (all at once, a wavefront stood still until the load unit's queue had room: 1 to 2 % of a large product)
  auto multiply = [&](int c, int h, bool loads) {
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const u32x4 wv = h == 0 ? codes8<F16>(wr[c][j][0], wr[c][j][1]) : codes8<F16>(wr[c][j][2], wr[c][j][3]);
#pragma unroll
      for (int i = 0; i < TM; ++i) tile[i][j] = product<F16>(xr[h][i], wv, c == 0 && h == 0 ? zero : tile[i][j]);
      if (loads) {
#pragma unroll
        for (int i = L * j / TN; i < L * (j + 1) / TN; ++i) issue(i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  const int mine = T::PERSIST ? (total - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x : 1;
  left = mine * stages;
  start();
#pragma unroll
  for (int s = 0; s < SLOTS; ++s)
    if (left > 0) {
#pragma unroll
      for (int i = 0; i < L; ++i) issue(i);
    }
  if (mine * stages >= SLOTS) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((SLOTS - 1) * L) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  // Operands are read half a block of products ahead.  The barrier stands in front of a stage's last products: behind it
  // the next stage's first operands are read under them, and the place of this one may be filled again.
  int slot = 0;
  read_w(0, 0);
  read_x(0, 0, 0);
  int todo = mine * stages;                              // stages not multiplied
  for (int e = (int)blockIdx.x; ; e += (int)gridDim.x) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (SECTIONS)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0, i = 1; s < stages; ++i) {
      const int end = SECTIONS ? s + section + (i > sections - longer ? 1 : 0) : stages;
      for (; s < end; ++s) {
        const int next = slot + T::kStage == SLOTS * T::kStage ? 0 : slot + T::kStage;
        read_x(slot, 0, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, 0, false);
        __builtin_amdgcn_sched_barrier(0);
        read_w(slot, 1);
        read_x(slot, 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, 1, false);
        __builtin_amdgcn_sched_barrier(0);
        read_x(slot, 1, 1);
#pragma unroll
        for (int j = 0; j < TN; ++j) sc[j] = *reinterpret_cast<const float*>(lds + slot + slane + j * 64);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, 0, false);
        __builtin_amdgcn_sched_barrier(0);
        const bool more = left > 0;
        if (--todo > 0) {
          // the next stage has arrived, and everybody has read this one
          if (SLOTS > 2 && todo >= SLOTS - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((SLOTS - 2) * L) : "memory");
          else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
          read_w(next, 0);
          read_x(next, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, 1, more);
        const int at = s + turned < stages ? s + turned : s + turned - stages;
        if (WK == 1 || b0 + at * WK + wk < b1) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int v = 0; v < 4; ++v) acc[i][j][v] = fmaf(sc[j], tile[i][j][v], acc[i][j][v]);
        }
        slot = next;
      }
      if constexpr (SECTIONS)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            sum[i][j] += acc[i][j];
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          }
    }
    if constexpr (SECTIONS)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j];
    if (!T::PERSIST) __syncthreads();                    // the last stage is read: its place is free

    constexpr int TO = TM / WK;                          // row tiles this wavefront stores
    static_assert(TO * WK == TM, "whole row tiles");
    if (WK == 2) {
      f32x4* const swap = reinterpret_cast<f32x4*>(smem) + (size_t)(wave % (WM * WN)) * (2 * TO * TN * 64);
#pragma unroll
      for (int i = 0; i < TO; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) swap[((wk * TO + i) * TN + j) * 64 + lane] = wk == 0 ? acc[TM - TO + i][j] : acc[i][j];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TO; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const f32x4 other = swap[(((1 - wk) * TO + i) * TN + j) * 64 + lane];
          acc[i][j] = wk == 0 ? acc[i][j] + other : other + acc[TM - TO + i][j];
        }
      __syncthreads();
    }

    // Register v of a tile holds row 4 * quad + v, column l16: 16 rows at a time go through LDS, so that they leave in
    // 16-byte stores of whole rows.
    int m0, n0;
    place(e, m0, n0);
    const int mw = m0 + wm + wk * TO * 16, nw = n0 + wn;
    float* const rows = reinterpret_cast<float*>(lds + (T::PERSIST ? SLOTS * T::kStage : 0)) + wave * 16 * PITCH;
    auto store = [&](auto* out, auto convert) {
      typedef decltype(convert(0.0f)) E;
      constexpr int V = 16 / sizeof(E);
      typedef E __attribute__((ext_vector_type(V))) vec;
#pragma unroll
      for (int i = 0; i < TO; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) rows[(4 * quad + v) * PITCH + j * 16 + l16] = acc[i][j][v];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int e = lane; e < 16 * TN * 16 / V; e += 64) {
          const int row = e / (TN * 16 / V), col = e % (TN * 16 / V) * V;
          const int m = mw + i * 16 + row;
          if (m >= p.m) continue;
          vec r;
#pragma unroll
          for (int v = 0; v < V; ++v) r[v] = convert(rows[row * PITCH + col + v]);
          E* dst = out + (size_t)m * p.n + nw + col;
          if (nw + col + V <= p.n) {
            __builtin_memcpy(dst, &r, 16);               // (rows of odd lengths begin anywhere; such stores one value at a time cost 1 us a call)
          } else {
#pragma unroll
            for (int v = 0; v < V; ++v)
              if (nw + col + v < p.n) dst[v] = r[v];
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    };
    if (p.k_splits > 1) store(p.partial + (size_t)blockIdx.y * split_step(p.m, p.n), [](float v) { return v; });
    else if (p.out_dtype == CPPMEGA_MI355_BF16) store((unsigned short*)p.out, f32_to_bf16_bits);
    else if (p.out_dtype == CPPMEGA_MI355_F16) store((unsigned short*)p.out, f32_to_f16_bits);
    else store((float*)p.out, [](float v) { return v; });
    if (!T::PERSIST || todo == 0) break;
  }
}

// out[m][n] = sum over the K splits of partial[split][m][n], in pairs.  Bound by latency (7 MB at 32 x 7168 x 8
// splits): with the splits' loads one after the other and stores of single values a call took 2 to 3 us longer.  Splits
// begin at whole 16-byte pieces, so that products of odd sizes are read alike (19 x 333 of 16 splits: 12 -> 4 us).  Code of
// its own for each number of splits: with a test in front of each load the first was waited for before the others were asked for.
template <int SPLITS>
__global__ __launch_bounds__(256) void fp8_gemm_reduce_kernel(const VecmatParams p) {
  const size_t total = (size_t)p.m * p.n, step = split_step(p.m, p.n);
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= total) return;
  f32x4 part[SPLITS];
#pragma unroll
  for (int z = 0; z < SPLITS; ++z) part[z] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.partial + (size_t)z * step + i));
#pragma unroll
  for (int step_z = 1; step_z < SPLITS; step_z *= 2)
#pragma unroll
    for (int z = 0; z + step_z < SPLITS; z += 2 * step_z) part[z] += part[z + step_z];
  const f32x4 s = part[0];
  if (i + 4 <= total && p.out_dtype != CPPMEGA_MI355_F32 && ((uintptr_t)p.out & 7) == 0) {
    const bool bf16 = p.out_dtype == CPPMEGA_MI355_BF16;
    *reinterpret_cast<uint2*>((unsigned short*)p.out + i) = bf16 ? make_uint2(pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]))
                                                                 : make_uint2(pack_f16(s[0], s[1]), pack_f16(s[2], s[3]));
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (i + v < total) store_as(p.out, i + v, p.out_dtype, s[v]);
  }
}

typedef Tile<2, 2, 1, 4, 2, 3, false> Tile32;            // 32 x 128, two groups, 150 KB of LDS
typedef Tile<2, 2, 1, 4, 1, 4, false> Tile32Short;       // 32 x 128, one group and up to four blocks, all on their way at once, 100 KB
typedef Tile<4, 2, 1, 4, 2, 2, false> Tile64Pair;        // 64 x 128, two groups, 132 KB
typedef Tile<4, 2, 1, 4, 1, 2, false> Tile64;            // 64 x 128, 66 KB: two workgroups on a CU, whose ends overlap
typedef Tile<4, 2, 1, 4, 1, 2, true> Tile64Many;         // the same, tile after tile
typedef Tile<4, 4, 2, 4, 1, 2, false> Tile256;           // 128 x 256, 132 KB

// What a tile shape costs, measured on MI355X: microseconds per stage with 1 and 2 of its workgroups on a CU, and per
// workgroup for its first loads and its stores.
enum Shape { kTile32, kTile32Short, kTile64Pair, kTile64, kTile64Many, kTile256 };
struct TileCost {
  int bm, bn, per_cu, groups;
  double stage_us[2], ends_us;
};
constexpr TileCost kCosts[] = {
    {32, 128, 1, 2, {1.145, 0.0}, 1.32},
    {32, 128, 1, 1, {0.8, 0.0}, 2.0},
    {64, 128, 1, 2, {1.21, 0.0}, 2.72},
    {64, 128, 2, 1, {0.92, 1.0}, 3.08},
    {64, 128, 2, 1, {0.5, 1.09}, 0.88},
    {128, 256, 1, 1, {1.71, 0.0}, 3.2},
};
constexpr int kSplits[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16};

struct GemmPlan { Shape shape; int splits; };

size_t split_bytes(int splits, int m, int n) { return splits > 1 ? splits * split_step(m, n) * sizeof(float) : 0; }

// The tile shape and K split with the smallest estimate: rounds of workgroups over the CUs, no less than the weights'
// stream takes, plus, for a split, one more launch and the partial sums written and read (8 bytes per sum).
// Fitted at 110 shapes of 17..4000 x 256..16400 x 512..16384, both scale layouts: the choice is 0.2 % from the best of all
// combinations there in the mean and 5 % at most.
// Float32 results over up to four blocks are one chain: the sum of two groups' sums is a rounding more (rms error against float64 1.13 x
// over 2 blocks, 1.08 x over 3, 1.02 x over 4).  Tiles of 32 rows with all their blocks on their way at once are as fast there (two groups /
// here: 83 x 763 x 256 4.5 / 4.3 us, 394 x 984 x 512 5.4 / 5.4, 102 x 9598 x 384 6.5 / 6.3, 2698 x 584 x 512 7.2 / 7.7).  Seven splits are for
// the largest tile, which keeps no second sum: in six its sums were longer (1434 x 719 x 16256 1.03 x the error, 49.7 us for 47.4).
// Splits whose sums need more than `have` bytes are left out; one split needs none.  64 x 128 tiles that are more than
// two to a CU are taken one after the other by as many workgroups (717 x 7411 x 1024: 23.7 -> 21.2 us, 1647 x 8297 x 1152:
// 46.3 -> 42.8; with one tile to a workgroup the loop costs 1 to 5 %).
GemmPlan gemm_plan(int m, int n, int k, bool f32, size_t have) {
  const int blocks = k / 128, cus = device_cus();
  GemmPlan best = {kTile32, 1};
  double best_us = 1e30;
  for (int shape = kTile32; shape <= kTile256; ++shape) {
    const TileCost& c = kCosts[shape];
    const long long tiles = (long long)((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
    const bool many = tiles > 2LL * cus;
    if ((shape == kTile64 && many) || (shape == kTile64Many && !many)) continue;
    const bool one_chain = f32 && blocks <= 4;
    if (one_chain ? c.groups > 1 : shape == kTile32Short) continue;
    for (int splits : kSplits) {
      if (splits > 1 && (splits * 2 > blocks || split_bytes(splits, m, n) > have || shape == kTile64Many)) break;
      if (splits == 7 && shape != kTile256) continue;
      const long long on_cu = (tiles * splits + cus - 1) / cus, rounds = on_cu / c.per_cu, rest = on_cu % c.per_cu;
      const int stages = ((blocks + splits - 1) / splits + c.groups - 1) / c.groups;
      double us = (double)rounds * (stages * c.stage_us[c.per_cu - 1] + c.ends_us);
      if (rest) us += stages * c.stage_us[0] + c.ends_us;
      const double stream_us = (double)n * k / 5.6e6 + 2.0;
      if (us < stream_us) us = stream_us;
      if (splits > 1) us += 4.8 + (double)splits * m * n * 8.0 / 5.5e6;
      if (us < best_us) { best_us = us; best = {(Shape)shape, splits}; }
    }
  }
  return best;
}

template <class T>
void launch_as(int m, int n, hipStream_t stream, const VecmatParams& p) {
  unsigned tiles = (unsigned)((m + T::BM - 1) / T::BM) * (unsigned)((n + T::BN - 1) / T::BN);
  if (T::PERSIST) {
    const unsigned most = (unsigned)(2 * device_cus()) & ~7u;          // a multiple of the XCDs
    if (most > 0 && tiles > most) tiles = most;
  }
  const dim3 grid(tiles, (unsigned)p.k_splits), block(T::kThreads);
  constexpr bool kSections = T::TM * T::TN <= 8 && T::SLOTS < 4;       // (the largest tile has no registers for a second sum, four blocks need none)
  const bool f16 = p.x_dtype == CPPMEGA_MI355_F16;
  if (kSections && p.out_dtype == CPPMEGA_MI355_F32) {
    if (f16) hipLaunchKernelGGL((fp8_gemm_kernel<T, true, kSections>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((fp8_gemm_kernel<T, false, kSections>), grid, block, 0, stream, p);
  } else if (f16) {
    hipLaunchKernelGGL((fp8_gemm_kernel<T, true, false>), grid, block, 0, stream, p);
  } else {
    hipLaunchKernelGGL((fp8_gemm_kernel<T, false, false>), grid, block, 0, stream, p);
  }
}

void launch_reduce(const VecmatParams& p, hipStream_t stream) {
  const size_t quads = ((size_t)p.m * p.n + 3) / 4;
  const unsigned threads = quads <= 65536 ? 64 : 256;
  const dim3 grid((unsigned)((quads + threads - 1) / threads)), block(threads);
  switch (p.k_splits) {                                         // (one of kSplits)
    case 2: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<2>, grid, block, 0, stream, p); break;
    case 3: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<3>, grid, block, 0, stream, p); break;
    case 4: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<4>, grid, block, 0, stream, p); break;
    case 5: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<5>, grid, block, 0, stream, p); break;
    case 6: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<6>, grid, block, 0, stream, p); break;
    case 7: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<7>, grid, block, 0, stream, p); break;
    case 8: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<8>, grid, block, 0, stream, p); break;
    case 10: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<10>, grid, block, 0, stream, p); break;
    case 12: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<12>, grid, block, 0, stream, p); break;
    default: hipLaunchKernelGGL(fp8_gemm_reduce_kernel<16>, grid, block, 0, stream, p); break;
  }
}

}  // namespace

// 5 to 16 rows stay with the kernel without staging while a CU has one workgroup of its 32 weight rows: with two it takes twice as long
// (16 rows, that kernel / this one: 8192 x 4096 10.3 / 11.4 us, 8500 x 1024 8.0 / 6.8, 8500 x 4096 17.3 / 12.0, 8500 x 16384 47.7 / 29.6, 16384 x
// 4096 19.3 / 16.1).  Measured at 5 .. 16 rows x 8400 .. 16400 x 512 .. 15900 with either layout of block scales: fewer than 12 rows gain
// from about 3000 channels on (5 x 8400 x 1024 0.86 x, 6 x 10300 x 2048 0.95, 4096 1.2); where three K splits of the tiles are more
// than the CUs and two leave some idle, up to 8192 channels (7 x 15814 x 14848 0.92), fewer with a scale per row, whose four
// bytes take a line of the cache each (6 x 12200 x 8192 0.97, 4096 1.20; 11 x 11467 x 7168 0.92), and any number where neither counts (11 x 14832 x 15872 1.12).  Float32 results stay there:
// one chain of sums here is up to 1.06 times as far from float64 as that kernel's (0.93 .. 1.06 of 5.7e-8 .. 1.0e-7), which results of 16 bits
// do not show.
static bool few_rows_here(const cppmega_mi355_vecmat_args_t& a) {
  const int cus = device_cus();
  if (a.m < 5 || a.n <= 32 * cus || (a.m < 12 && a.k < 3072) || a.out_dtype == CPPMEGA_MI355_F32) return false;
  const bool row_scales = a.scale_w_kind == CPPMEGA_MI355_WSCALE_ROW_BLOCK;
  if ((a.n + 127) / 128 * 3 <= cus || (a.m >= 9 && !row_scales)) return true;
  return a.k <= (row_scales ? 6144 : 8192);
}

// bf16 / fp16 activations, whole 128-channel blocks, more rows than the kernels without staging take
bool fp8_gemm_shape(const cppmega_mi355_vecmat_args_t& a) {
  return (a.x_dtype == CPPMEGA_MI355_BF16 || a.x_dtype == CPPMEGA_MI355_F16) && (a.m > 16 || few_rows_here(a)) && a.k % 128 == 0 &&
         a.k <= (1 << 22);                                      // a tile's rows within 32-bit offsets
}

size_t fp8_gemm_workspace_bytes(const cppmega_mi355_vecmat_args_t& a) {
  int splits = gemm_plan(a.m, a.n, a.k, a.out_dtype == CPPMEGA_MI355_F32, SIZE_MAX).splits;
  // A few small tiles ask for the room of three splits (3 MB at most) where the plan has one or two: as much as when each of them was
  // split, so that scratch laid out by asking for one such size goes on serving the others.
  if (splits < 3 && a.k >= 6 * 128 && (long long)((a.m + 31) / 32) * ((a.n + 127) / 128) <= device_cus() / 4) splits = 3;
  return split_bytes(splits, a.m, a.n);
}

int fp8_gemm_launch(VecmatParams p, size_t workspace_bytes, hipStream_t stream) {
  // (the sums of splits are read in 16-byte pieces)
  const GemmPlan g = gemm_plan(p.m, p.n, p.k, p.out_dtype == CPPMEGA_MI355_F32, ((uintptr_t)p.partial & 15) == 0 ? workspace_bytes : 0);
  p.k_splits = g.splits;
  const long long tiles = (long long)((p.m + kCosts[g.shape].bm - 1) / kCosts[g.shape].bm) * ((p.n + kCosts[g.shape].bn - 1) / kCosts[g.shape].bn);
  if (tiles > 0x7fffffffLL) return fail(CPPMEGA_MI355_ERR_SHAPE, "vecmat: M=%d N=%d has too many tiles", p.m, p.n);
  switch (g.shape) {
    case kTile32: launch_as<Tile32>(p.m, p.n, stream, p); break;
    case kTile32Short: launch_as<Tile32Short>(p.m, p.n, stream, p); break;
    case kTile64Pair: launch_as<Tile64Pair>(p.m, p.n, stream, p); break;
    case kTile64: launch_as<Tile64>(p.m, p.n, stream, p); break;
    case kTile64Many: launch_as<Tile64Many>(p.m, p.n, stream, p); break;
    case kTile256: launch_as<Tile256>(p.m, p.n, stream, p); break;
  }
  CM_HIP_CHECK(hipGetLastError());
  if (g.splits > 1) {
    launch_reduce(p, stream);
    CM_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

}  // namespace cm
