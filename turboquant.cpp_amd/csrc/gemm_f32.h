// What the 32-bit path's products share: the arguments of a product and its bias.
#pragma once
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct F32GemmArgs {
  const float* a;
  int64_t lda;
  const int* a_rows;       // row of `a` that feeds output row m (-1: none), or null for m itself
  int a_gather;            // 0: a_rows only marks live rows (>= 0) and row m itself is read
  const float* w;          // [groups][N][K]
  const float* w2;         // second matrix of the gated pair, or null
  int64_t group_stride;
  const int* tile_group;   // group of each row tile, or null (group 0)
  const int* n_tiles;      // number of live row tiles on the device, or null (all)
  const void* bias;
  int bias_type;
  float* out;
  int64_t ldc;
  int M, N, K;
  int gate;                // activation of the gated pair
  float limit;             // of the gated pair (gated_pair in common.h); 0: none
};

__device__ __forceinline__ float f32_bias_at(const F32GemmArgs& g, int n) {
  if (!g.bias) return 0.f;
  return g.bias_type == TQ_F32 ? ((const float*)g.bias)[n] : to_f32(((const bf16_t*)g.bias)[n]);
}

// gemm_f32_split.hip: a product of more than 64 rows (or over experts with units of 64 rows; `pairs`: two units at a
// time, by the items behind the row tiles) on the bfloat16 instructions, k in runs whose sums go to `part` if there is
// more than one.
int f32_split_runs(int M, int N, int K, int* k_per_run);
int f32_split_product(const F32GemmArgs& g, bool pairs, int runs, int k_per_run, float* part, hipStream_t st);
