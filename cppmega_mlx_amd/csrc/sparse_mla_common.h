// Parameter block shared by the sparse-MLA kernels.
#pragma once

#include "common.h"

namespace cm {

struct MlaParams {
  const void* q;
  const void* q_scale;
  const void* kv;
  const void* kv_scale;
  const void* rope;
  const void* indices;
  const float* sinks;
  void* out;
  float* lse;
  void* workspace;
  float* scores;        // score-only entry point: [B, S, H, topk] fp32
  int q_dtype, q_scale_kind, q_scale_block;
  int kv_dtype, kv_scale_kind, kv_scale_block;
  int rope_dtype, rope_dim;
  int index_dtype, out_dtype;
  int B, S, H, G, Skv, topk;
  int d_qk, d_kv, d_v;
  int heads_per_group;
  int num_splits;       // split-KV factor of the MFMA kernel
  int keys_per_split;
  int heads_per_wg;     // 0: 32-head tile kernel; 32 or 64: a producer/consumer kernel (sparse_mla_latent.hip, sparse_mla_rows16.hip)
  int plan_level;       // how the launch is planned: see sparse_mla_mfma_plan_within
  int rows16;           // with heads_per_wg: the kernel for 16-bit rows
  int few;              // with heads_per_wg: the kernel of workgroups of 16 heads (sparse_mla_few.hip)
  int no_few;           // the scratch does not hold that kernel's plan: plans without it
  int tile_sharing;     // tile kernel on 16-bit rows: the 4 wavefronts take 4 head groups over one key stream
  float sm_scale;
  const float* sm_scale_dev;     // device copy of the softmax scale; read in place of sm_scale when set
  const int* has_sinks_dev;      // device flag; sinks are ignored when it is set and holds 0
  int Skv_pitch;                 // key rows between two batches of the cache buffers (>= Skv)
};

// softmax scale and sink switch as the kernels read them (uniform loads)
__device__ __forceinline__ float mla_sm_scale(const MlaParams& p) { return p.sm_scale_dev ? *p.sm_scale_dev : p.sm_scale; }
__device__ __forceinline__ bool mla_has_sinks(const MlaParams& p) {
  return p.sinks != nullptr && (p.has_sinks_dev == nullptr || *p.has_sinks_dev != 0);
}

__device__ __forceinline__ long long load_index(const MlaParams& p, size_t i) {
  return p.index_dtype == CPPMEGA_MI355_I64 ? ((const long long*)p.indices)[i]
                                            : (long long)((const int*)p.indices)[i];
}

// scale of element block `blk` of row `row` (row = flattened leading index)
__device__ __forceinline__ float row_scale(const void* scale, int kind, size_t row, int nblk, int blk) {
  switch (kind) {
    case CPPMEGA_MI355_SCALE_PER_TOKEN: return ((const float*)scale)[row];
    case CPPMEGA_MI355_SCALE_E8M0: return e8m0_to_f32(((const unsigned char*)scale)[row * nblk + blk]);
    case CPPMEGA_MI355_SCALE_F32_BLOCK: return ((const float*)scale)[row * nblk + blk];
    default: return 1.0f;
  }
}

int sparse_mla_scalar_launch(const MlaParams& p, hipStream_t stream);
int sparse_mla_scores_launch(const MlaParams& p, hipStream_t stream);
int sparse_mla_mfma_launch(const MlaParams& p, hipStream_t stream);
bool sparse_mla_mfma_supported(const MlaParams& p);
size_t sparse_mla_mfma_workspace_bytes(const MlaParams& p);
void sparse_mla_mfma_plan(MlaParams& p);
// The plan for a caller who brings `have` bytes of workspace, and what it needs: the fastest one (level 0, what the
// size query answers) if that fits (first with, then without the kernel of 16 heads where there are more), else key splits only until 256 workgroups are there and no copy of the cache
// (level 1), else the kernel of sparse_mla_mfma.hip where it serves the shape (level 2).
size_t sparse_mla_mfma_plan_within(MlaParams& p, size_t have);

// partial values that a key split keeps of 32 heads: [4 groups of 128 channels][8 row pairs][64 lanes][8]
constexpr int kMlaPartFloats = 4 * 16 * 64 * 4;
int sparse_mla_combine_f32(const MlaParams& p, hipStream_t stream);    // merges the key splits' float32 partial values

// Key splits of the producer/consumer kernels, whose workgroups have a CU to themselves: the number (up to 16, up to
// max_keys each) with the least modelled time - whole rounds of 256 workgroups, each with its workgroups' start and end
// and tile_us per tile of 32 keys, then, with several splits, the merging kernel and the traffic of the sums of `heads`
// heads per workgroup, written and read.
// `narrow`: the sums are bfloat16, so there are no more splits than doubling until 256 workgroups are there makes.
// At plan level 1: the doubled number.
// Returns the modelled microseconds (level 0).
double mla_key_splits(MlaParams& p, long long units, int max_keys, double tile_us, int heads, bool narrow);

// producer/consumer kernel for 16-bit rows (sparse_mla_rows16.hip); dispatched by the *_mfma_* functions
bool sparse_mla_rows16_supported(const MlaParams& p);
double sparse_mla_rows16_plan(MlaParams& p);             // modelled microseconds
// E8M0 rows: room for a bfloat16 copy of the queries and of every cache row (0: not such rows), and the launch that writes it to the
// workspace and makes p the same call on 16-bit rows, with the workspace behind the copy
size_t sparse_mla_e8m0_copy_bytes(const MlaParams& p);
int sparse_mla_e8m0_copy(MlaParams& p, hipStream_t stream);
int sparse_mla_rows16_launch(const MlaParams& p, hipStream_t stream);   // includes its combine step
size_t sparse_mla_rows16_workspace_bytes(const MlaParams& p);

// kernel of workgroups of 16 heads (sparse_mla_few.hip); dispatched by the *_mfma_* functions
bool sparse_mla_few_supported(const MlaParams& p);
void sparse_mla_few_plan(MlaParams& p);
int sparse_mla_few_launch(const MlaParams& p, hipStream_t stream);     // includes its combine step
size_t sparse_mla_few_workspace_bytes(const MlaParams& p);

// shared-tile kernel for FP8 latent caches (sparse_mla_latent.hip); dispatched by the *_mfma_* functions
bool sparse_mla_latent_supported(const MlaParams& p);
bool sparse_mla_latent_only(const MlaParams& p);         // no other kernel has served these shapes
double sparse_mla_latent_plan(MlaParams& p);             // modelled microseconds
int sparse_mla_latent_launch(const MlaParams& p, hipStream_t stream);   // includes its combine step
size_t sparse_mla_latent_workspace_bytes(const MlaParams& p);

}  // namespace cm
