// FP8 (e4m3) block-scaled weight GEMM for batches and prefill chunks (gfx950).
//
//   out[m, n] = sum_k dec(w[n, k]) * w_scale(n, k / 128) * x[m, k],   x bf16 or fp16, fp32 accumulation
//
// The kernels of fp8_vecmat.hip read the whole weight once per 4 to 16 activation rows; from 17 rows on a
// tile of both operands is worth staging in LDS.  Measured (microseconds, against passes over the weights):
// M x N x K = 2048 x 8192 x 1536: 66 (3364), 48 x 7168 x 16384: 38 (60), 300 x 1434 x 896: 10 (190),
// 2048 x 7168 x 16384: 490 = 980 TFLOP/s.  What bounds it: a large product, the issue of MFMAs and of the
// vector instructions between them (128 per 32 MFMAs: conversions and scaled sums); a short one (K = 1536),
// the first loads and the stores of a tile, 10 of 33 us, which a CU with one workgroup does not overlap; a
// small batch, the weight stream (32 x 7168 x 16384: 37.5 us a call, 3.1 TB/s).

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
__device__ __forceinline__ f32x16 product(const u32x4& a, const u32x4& b, const f32x16& c) {
  if (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Slot of 16-byte piece `piece` of row `row` in an LDS tile of `PIECES` pieces per row.  A 16-byte read
// is served sixteen lanes (256 bytes, all banks) at a time, and the rows of such a group differ in their
// low bits: the exclusive-or spreads one piece of 16 rows over the 16 bank groups.
template <int PIECES>
__device__ __forceinline__ int slot(int row, int piece) {
  return row * PIECES + (piece ^ ((row / (16 / PIECES)) & (PIECES - 1)));
}

// TM x TN tiles of 32 x 32 per wavefront, WM x WN wavefronts, BK channels per stage.
//
// Every 128-channel block is accumulated from zero and enters the sums as acc += scale * tile, so fp32
// scales of any kind are applied exactly; in the product layout (weights as the second operand) a lane
// holds one output channel, i.e. one scale per tile.  A lane's 16 weight bytes feed two products: the
// contraction runs over the channels in the order the bytes lie in, and the activation pieces follow it.
template <int TM, int TN, int WM, int WN, int BK, bool F16>
__global__ __launch_bounds__(64 * WM * WN, 2) void fp8_gemm_kernel(const VecmatParams p) {
  constexpr int kGemmThreads = 64 * WM * WN;
  constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
  constexpr int XP = BK / 8, WP = BK / 16;               // 16-byte pieces per row of the two tiles
  constexpr int XL = BM * XP / kGemmThreads, WL = BN * WP / kGemmThreads;
  static_assert(XL * kGemmThreads == BM * XP && WL * kGemmThreads == BN * WP, "whole pieces per thread");
  constexpr int STEPS = 128 / BK;
  constexpr int PITCH = TN * 32 + 4;                     // of the rows on their way out
  constexpr int TILES = 2 * (BM * XP + BN * WP), ROWS = WM * WN * 32 * PITCH / 4;
  __shared__ u32x4 smem[TILES > ROWS ? TILES : ROWS];
  u32x4* const xs = smem;                                // [2][BM * XP]
  u32x4* const ws = smem + 2 * BM * XP;                  // [2][BN * WP]

  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave / WN) * TM * 32, wn = (wave % WN) * TN * 32;
  const int half = lane >> 5, l32 = lane & 31;

  // Tile of this workgroup.  Consecutive workgroups go round the eight XCDs: every XCD takes one run of
  // the order (groups of eight column tiles; inside, row tile by row tile), so that its L2 holds the
  // weights of a group while the row tiles pass.
  const int tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  const int q = total >> 3, r = total & 7, xcd = (int)blockIdx.x & 7;
  const int t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + ((int)blockIdx.x >> 3);
  const int per_group = tiles_m * 8, group = t / per_group;
  const int width = tiles_n - group * 8 < 8 ? tiles_n - group * 8 : 8;
  const int in_group = t - group * per_group;
  const int m0 = (in_group / width) * BM, n0 = (group * 8 + in_group % width) * BN;

  const int blocks = p.k / 128;
  const int b0 = (int)((long long)blocks * blockIdx.y / p.k_splits), b1 = (int)((long long)blocks * (blockIdx.y + 1) / p.k_splits);

  // one uniform base per operand, moved on by a stage at a time, and 32-bit lane offsets
  const char* xbase = reinterpret_cast<const char*>(p.x) + ((size_t)m0 * p.k + (size_t)b0 * 128) * 2;
  const char* wbase = reinterpret_cast<const char*>(p.w) + (size_t)n0 * p.k + (size_t)b0 * 128;
  unsigned xoff[XL], woff[WL];
  int xslot[XL], wslot[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int e = tid + i * kGemmThreads, row = e / XP, piece = e % XP;
    const int m = m0 + row < p.m ? row : p.m - 1 - m0;       // rows past the end repeat the last one and are not stored
    xoff[i] = (unsigned)m * (unsigned)p.k * 2u + (unsigned)piece * 16u;
    xslot[i] = slot<XP>(row, piece);
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int e = tid + i * kGemmThreads, row = e / WP, piece = e % WP;
    const int n = n0 + row < p.n ? row : p.n - 1 - n0;
    woff[i] = (unsigned)n * (unsigned)p.k + (unsigned)piece * 16u;
    wslot[i] = slot<WP>(row, piece);
  }
  const float* sg[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 32 + l32 < p.n ? n0 + wn + j * 32 + l32 : p.n - 1;
    sg[j] = p.scale_w + (size_t)(n >> p.srow_shift) * p.srow_stride;
  }

  // Two register sets, so that two stages are on their way while one computes out of LDS and one is
  // written there.  Loads in the loop are unconditional (behind a branch the compiler waits for them at
  // once): past the last stage they fetch it again.
  u32x4 xr[2][XL], wr[2][WL];
  const int stages = (b1 - b0) * STEPS;
  int fetched = 0;
  auto fetch = [&](int set) {
#pragma unroll
    for (int i = 0; i < XL; ++i) xr[set][i] = *reinterpret_cast<const u32x4*>(xbase + xoff[i]);
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      // one row tile: the weights pass once and need not stay in the caches
      const u32x4* src = reinterpret_cast<const u32x4*>(wbase + woff[i]);
      wr[set][i] = WM == 1 ? __builtin_nontemporal_load(src) : *src;
    }
    const bool more = ++fetched < stages;
    xbase += more ? BK * 2 : 0;
    wbase += more ? BK : 0;
  };
  auto stage = [&](int set, int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) xs[buf * BM * XP + xslot[i]] = xr[set][i];
#pragma unroll
    for (int i = 0; i < WL; ++i) ws[buf * BN * WP + wslot[i]] = wr[set][i];
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // operands of one 32-channel step
  struct Operands { u32x4 w[TN], x[TM][2]; };
  auto read = [&](int buf, int kk, Operands& o) {
#pragma unroll
    for (int j = 0; j < TN; ++j) o.w[j] = ws[buf * BN * WP + slot<WP>(wn + j * 32 + l32, kk * 2 + half)];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) o.x[i][h] = xs[buf * BM * XP + slot<XP>(wm + i * 32 + l32, kk * 4 + half * 2 + h)];
  };
  Operands ops[2];
  // One stage out of LDS buffer `buf`, operands read a step ahead.  The barrier stands in front of the
  // stage's last products: behind it the next stage's first operands can be read under them.  (The other
  // buffer was last read in front of the previous stage's barrier.)
  auto step = [&](int buf, f32x16 (&tile)[TM][TN]) {
    constexpr int KK = BK / 32;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if (kk == KK - 1) {
        __syncthreads();
        read(buf ^ 1, 0, ops[0]);
      } else {
        read(buf, kk + 1, ops[(kk + 1) & 1]);
      }
      if (kk == 0) {
        stage(buf ^ 1, buf ^ 1);
        fetch(buf ^ 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      const Operands& o = ops[kk & 1];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const u32x4 wv = h == 0 ? codes8<F16>(o.w[j][0], o.w[j][1]) : codes8<F16>(o.w[j][2], o.w[j][3]);
#pragma unroll
          for (int i = 0; i < TM; ++i) tile[i][j] = product<F16>(o.x[i][h], wv, tile[i][j]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // one 128-channel block: STEPS stages from LDS buffer `buf` on
  auto block = [&](int b, int buf) {
    f32x16 tile[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) tile[i][j][v] = 0.0f;
    float sc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) sc[j] = sg[j][(size_t)b * p.scol_stride];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) step((buf + s) & 1, tile);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = fmaf(sc[j], tile[i][j][v], acc[i][j][v]);
  };

  fetch(0);
  stage(0, 0);
  fetch(1);
  fetch(0);
  __syncthreads();
  read(0, 0, ops[0]);
  int b = b0;
  if (STEPS == 1) {
    for (; b + 2 <= b1; b += 2) {
      block(b, 0);
      block(b + 1, 1);
    }
    if (b < b1) block(b, 0);
  } else {
    for (; b < b1; ++b) block(b, 0);
  }

  // Register v of a tile holds row 8 * (v / 4) + 4 * half + v % 4, column l32: 32 rows at a time go
  // through LDS, so that they leave in 16-byte stores of whole rows.
  float* const rows = reinterpret_cast<float*>(smem) + wave * 32 * PITCH;
  const int nw = n0 + wn;
  auto store = [&](auto* out, auto convert) {
    typedef decltype(convert(0.0f)) T;
    constexpr int V = 16 / sizeof(T);
    typedef T __attribute__((ext_vector_type(V))) vec;
    const bool vectors = p.n % V == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) rows[(8 * (v >> 2) + 4 * half + (v & 3)) * PITCH + j * 32 + l32] = acc[i][j][v];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int e = lane; e < 32 * TN * 32 / V; e += 64) {
        const int row = e / (TN * 32 / V), col = e % (TN * 32 / V) * V;
        const int m = m0 + wm + i * 32 + row;
        if (m >= p.m) continue;
        vec r;
#pragma unroll
        for (int v = 0; v < V; ++v) r[v] = convert(rows[row * PITCH + col + v]);
        T* dst = out + (size_t)m * p.n + nw + col;
        if (vectors) {
          if (nw + col < p.n) *reinterpret_cast<vec*>(dst) = r;
        } else {
#pragma unroll
          for (int v = 0; v < V; ++v)
            if (nw + col + v < p.n) dst[v] = r[v];
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  __syncthreads();                                       // the last stage is read
  if (p.k_splits > 1) store(p.partial + (size_t)blockIdx.y * p.m * p.n, [](float v) { return v; });
  else if (p.out_dtype == CPPMEGA_MI355_BF16) store((unsigned short*)p.out, f32_to_bf16_bits);
  else if (p.out_dtype == CPPMEGA_MI355_F16) store((unsigned short*)p.out, f32_to_f16_bits);
  else store((float*)p.out, [](float v) { return v; });
}

// out[m][n] = sum over the K splits of partial[split][m][n], in split order.  Bound by latency (7 MB at 32 x 7168 x 8
// splits): with the splits' loads one after the other and stores of single values a call took 2 to 3 us longer.
__global__ __launch_bounds__(256) void fp8_gemm_reduce_kernel(const VecmatParams p) {
  const size_t total = (size_t)p.m * p.n;
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  if ((total & 3) == 0) {
    // (the loads of the up to 16 splits are in flight together)
    f32x4 part[16], s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int z = 0; z < 16; ++z)
      if (z < p.k_splits) part[z] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.partial + (size_t)z * total + i));
#pragma unroll
    for (int z = 0; z < 16; ++z)
      if (z < p.k_splits) s += part[z];
    if (p.out_dtype != CPPMEGA_MI355_F32 && ((uintptr_t)p.out & 7) == 0) {
      const bool bf16 = p.out_dtype == CPPMEGA_MI355_BF16;
      *reinterpret_cast<uint2*>((unsigned short*)p.out + i) = bf16 ? make_uint2(pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]))
                                                                   : make_uint2(pack_f16(s[0], s[1]), pack_f16(s[2], s[3]));
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) store_as(p.out, i + v, p.out_dtype, s[v]);
    }
  } else {
    for (size_t e = i; e < i + 4 && e < total; ++e) {
      float s = 0.0f;
      for (int z = 0; z < p.k_splits; ++z) s += p.partial[(size_t)z * total + e];
      store_as(p.out, e, p.out_dtype, s);
    }
  }
}

// What a tile shape costs, measured on MI355X: microseconds per 128-channel block with 1, 2, .. of its
// workgroups on a CU, and per workgroup for its first loads and its stores.
struct TileShape {
  int bm, bn, per_cu;
  double block_us[3], ends_us;
};
constexpr TileShape kShapes[] = {
    {32, 128, 3, {0.82, 1.48, 3.23}, 6.0},
    {64, 128, 2, {0.85, 1.77, 0.0}, 8.35},
    {128, 256, 1, {1.77, 0.0, 0.0}, 9.3},
};
constexpr int kSplits[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 16};

struct GemmPlan { const TileShape* shape; int splits; };

size_t split_bytes(int splits, int m, int n) { return splits > 1 ? (size_t)splits * m * n * sizeof(float) : 0; }

// The tile shape and K split with the smallest estimate: rounds of workgroups over the CUs, plus, for a
// split, one more launch and the partial sums written and read (8 bytes per sum).  Fitted to all combinations but
// those of 9 splits at 55 shapes of 17..1000 x 512..16384 x 896..16384: the choice is 0.4 % from the best of them in the
// mean and 7 % at most.  9 splits give 56 column tiles two workgroups on nearly every CU where 8 leave a quarter of the
// CUs with one (32 x 7168 x 16384: 41 -> 39 us, the calls of 13 .. 16 splits that finer steps would pick are no faster).  The third workgroup on a CU brings nothing (the weights' stream is what they share).
// Splits whose sums need more than `have` bytes are left out; one split needs none.
GemmPlan gemm_plan(int m, int n, int k, size_t have) {
  const int blocks = k / 128, cus = device_cus();
  GemmPlan best = {&kShapes[0], 1};
  double best_us = 1e30;
  for (const TileShape& s : kShapes) {
    const double tiles = (double)((m + s.bm - 1) / s.bm) * ((n + s.bn - 1) / s.bn);
    for (int splits : kSplits) {
      if (splits > 1 && (splits * 2 > blocks || split_bytes(splits, m, n) > have)) break;
      const long long wgs = (long long)tiles * splits, on_cu = (wgs + cus - 1) / cus;
      const double steps = (blocks + splits - 1) / splits;
      const long long rounds = on_cu / s.per_cu, rest = on_cu % s.per_cu;
      double us = (double)rounds * (steps * s.block_us[s.per_cu - 1] + s.ends_us);
      if (rest) us += steps * s.block_us[rest - 1] + s.ends_us;
      if (splits > 1) us += 3.3 + (double)splits * m * n * 8.0 / 5.1e6;
      if (us < best_us) { best_us = us; best = {&s, splits}; }
    }
  }
  return best;
}

template <int TM, int TN, int WM, int WN, int BK>
void launch_as(dim3 grid, hipStream_t stream, const VecmatParams& p) {
  const dim3 block(64 * WM * WN);
  if (p.x_dtype == CPPMEGA_MI355_F16) hipLaunchKernelGGL((fp8_gemm_kernel<TM, TN, WM, WN, BK, true>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((fp8_gemm_kernel<TM, TN, WM, WN, BK, false>), grid, block, 0, stream, p);
}

}  // namespace

// bf16 / fp16 activations, whole 128-channel blocks, more rows than the kernels without staging take
bool fp8_gemm_shape(const cppmega_mi355_vecmat_args_t& a) {
  return (a.x_dtype == CPPMEGA_MI355_BF16 || a.x_dtype == CPPMEGA_MI355_F16) && a.m > 16 && a.k % 128 == 0 &&
         a.k <= (1 << 22);                                      // a tile's rows within 32-bit offsets
}

size_t fp8_gemm_workspace_bytes(const cppmega_mi355_vecmat_args_t& a) {
  return split_bytes(gemm_plan(a.m, a.n, a.k, SIZE_MAX).splits, a.m, a.n);
}

int fp8_gemm_launch(VecmatParams p, size_t workspace_bytes, hipStream_t stream) {
  const GemmPlan g = gemm_plan(p.m, p.n, p.k, workspace_bytes);
  p.k_splits = g.splits;
  const long long tiles = (long long)((p.m + g.shape->bm - 1) / g.shape->bm) * ((p.n + g.shape->bn - 1) / g.shape->bn);
  if (tiles > 0x7fffffffLL) return fail(CPPMEGA_MI355_ERR_SHAPE, "vecmat: M=%d N=%d has too many tiles", p.m, p.n);
  const dim3 grid((unsigned)tiles, (unsigned)g.splits);
  if (g.shape->bm == 32) launch_as<1, 1, 1, 4, 128>(grid, stream, p);
  else if (g.shape->bm == 64) launch_as<2, 1, 1, 4, 128>(grid, stream, p);
  else launch_as<2, 2, 2, 4, 64>(grid, stream, p);
  CM_HIP_CHECK(hipGetLastError());
  if (g.splits > 1) {
    const size_t quads = ((size_t)p.m * p.n + 3) / 4;
    hipLaunchKernelGGL(fp8_gemm_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, stream, p);
    CM_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

}  // namespace cm
