// What the kernels of the gated delta rule share (delta_rule.hip, delta_chunks.hip): the sizes, and the functions of the gates.
#pragma once
#include "common.h"

struct DeltaDims {
  int H, G, D, V;         // heads, q/k heads, key width, value width
  int taps;               // of the convolution
  int ra, rg;             // ranks of the decay's and the gate's first product
  int mode;               // 0: a decay per head and key channel, behind low-rank products; 1: a decay per head (ra = rg = 0)
};
__host__ __device__ __forceinline__ int dd_channels(const DeltaDims& d) { return 2 * d.G * d.D + d.H * d.V; }
__host__ __device__ __forceinline__ int dd_np(const DeltaDims& d) {
  return d.mode == 1 ? dd_channels(d) + 2 * d.H + d.H * d.V : dd_channels(d) + d.H + d.ra + d.rg;
}
__host__ __device__ __forceinline__ int64_t dd_state(const DeltaDims& d) {
  return (int64_t)d.H * d.D * d.V + (int64_t)dd_channels(d) * (d.taps - 1);
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// The recurrence token by token over the runs of fewer than `below` tokens; ag is only read.
int delta_short_runs(const float* qn, const float* kn, const float* vc, const float* beta, const float* ag, const float* a_log,
                     const float* dt_bias, const int* cu_seqlens, const int* slots, float* state, int64_t state_stride,
                     const DeltaDims& d, int below, int T, int B, float* o_raw, hipStream_t st);
