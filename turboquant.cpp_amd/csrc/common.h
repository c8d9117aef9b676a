// Shared definitions of the gfx950 kernels.
//
// One library is built per activation type: TQ_ACT_BF16 (activations and cache in
// bfloat16, every sum in float) or TQ_ACT_F32 (everything in float, no matrix cores
// with reduced-precision inputs).  Weights carry their own type at run time
// (TQ_F32 or TQ_BF16) because a tensor that the checkpoint stores in 32 bits stays so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define TQ_F32 0
#define TQ_BF16 1

// error codes of the extern "C" entry points (0 = ok, > 0 = hipError_t)
#define TQ_ERR_BAD_ARG (-1)
#define TQ_ERR_UNSUPPORTED (-2)
// added to a tile_rows of 64 of a product over experts: the units that the row order's items hold, two or four of one
// expert, per workgroup (see tq_gemm_mfma)
#define TQ_TILE_PAIRS 1024
// added to the unit of the order of pairs by expert: its items hold four row tiles instead of two (see moe.hip).  Above every unit:
// a unit of rows may be any number whose rows fit the order.
#define TQ_ITEMS_OF_FOUR (1 << 30)
// The row order's n_tiles may hold more than its two numbers, 48 in all, of which the last 32, two runs of 16, are queues: written with the
// order (and the third, the experts that have rows) where TQ_ORDER_QUEUES is added to its unit of 64, each for one product (tile_rows with TQ_TILE_QUEUE added once or twice) behind it.
// The sign: no unit of rows has it, and with any other unit than 64 it stays a negative number, which is refused.
#define TQ_ORDER_QUEUES (-0x7fffffff - 1)
#define TQ_TILE_QUEUE 2048
#define TQ_GEMM_ACT_ALONE 256      // added to tq_gemm_mfma's gate: the activation of a plain product's result

struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }

// Round to nearest even; NaN stays NaN: one instruction, the bits of the rounding by integers (of all 2^32 floats), which took five.
__device__ __forceinline__ bf16_t f32_to_bf16(float f) { return {__builtin_bit_cast(uint16_t, (__bf16)f)}; }
// Two of them side by side, the first in the low half.
__device__ __forceinline__ uint32_t f32_to_bf16_pair(float lo, float hi) {
  typedef __bf16 pair __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, pair{(__bf16)lo, (__bf16)hi});
}

template <class T>
__device__ __forceinline__ T from_f32(float f);
template <>
__device__ __forceinline__ float from_f32<float>(float f) { return f; }
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float f) { return f32_to_bf16(f); }

#if defined(TQ_ACT_BF16)
typedef bf16_t act_t;
#define TQ_ACT_TYPE TQ_BF16
#elif defined(TQ_ACT_F32)
typedef float act_t;
#define TQ_ACT_TYPE TQ_F32
#else
#error "define TQ_ACT_BF16 or TQ_ACT_F32"
#endif

#define TQ_WAVE 64

// v and the value of lane l ^ O put together by f, for the whole wave.  In the vector unit throughout: a step of the shuffle that
// goes through LDS takes as long as twenty additions, and a short kernel of one token is made of such chains (a sum over a wave: 60
// clocks instead of 420).
template <int O, class F>
__device__ __forceinline__ float with_lane_xor(float v, F f) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "a power of two");
  if constexpr (O >= 16) {
    typedef unsigned two __attribute__((ext_vector_type(2)));
    const unsigned u = __float_as_uint(v);
    const two s = __builtin_bit_cast(two, O == 32 ? __builtin_amdgcn_permlane32_swap(u, u, false, false)
                                                  : __builtin_amdgcn_permlane16_swap(u, u, false, false));
    return f(__uint_as_float(s.x), __uint_as_float(s.y));      // one is the lane's own value, the other its partner's
  } else {
    const int i = __float_as_int(v);
    int o;
    if constexpr (O == 8) o = __builtin_amdgcn_update_dpp(i, i, 0x128, 0xf, 0xf, false);                 // row_ror:8
    else if constexpr (O == 4) o = __builtin_amdgcn_update_dpp(i, __builtin_amdgcn_update_dpp(i, i, 0x141, 0xf, 0xf, false), 0x1B, 0xf, 0xf, false);      // half mirror, then [3, 2, 1, 0]
    else if constexpr (O == 2) o = __builtin_amdgcn_update_dpp(i, i, 0x4E, 0xf, 0xf, false);             // [2, 3, 0, 1]
    else o = __builtin_amdgcn_update_dpp(i, i, 0xB1, 0xf, 0xf, false);                                   // [1, 0, 3, 2]
    return f(v, __int_as_float(o));
  }
}
// Over groups of L neighbouring lanes (L a power of two), from the halves down to the pairs.
template <int L, class F>
__device__ __forceinline__ float lanes_fold(float v, F f) {
  if constexpr (L > 1) {
    v = with_lane_xor<L / 2>(v, f);
    return lanes_fold<L / 2>(v, f);
  }
  return v;
}
struct LanesSum {
  __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct LanesMax {
  __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
__device__ __forceinline__ float wave_sum(float v) {
  return lanes_fold<TQ_WAVE>(v, LanesSum());
}
__device__ __forceinline__ float wave_max(float v) {
  return lanes_fold<TQ_WAVE>(v, LanesMax());
}

// Inclusive sum over the lanes up to one's own, in the vector unit as well: within rows of 16 by shifts, then the rows' last lanes
// into the rows behind them.
__device__ __forceinline__ int wave_scan_add(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);      // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);     // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);     // row_bcast:31 into rows 2 and 3
  return v;
}

// Sum over a workgroup in a fixed order: waves reduce by butterfly, wave totals are added
// in wave order.  `red` holds one float per wave.  Every thread gets the total.
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x / TQ_WAVE, lane = threadIdx.x % TQ_WAVE;
  const int nw = (blockDim.x + TQ_WAVE - 1) / TQ_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}
__device__ __forceinline__ float block_max(float v, float* red) {
  v = wave_max(v);
  const int wave = threadIdx.x / TQ_WAVE, lane = threadIdx.x % TQ_WAVE;
  const int nw = (blockDim.x + TQ_WAVE - 1) / TQ_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = red[0];
  for (int i = 1; i < nw; ++i) t = fmaxf(t, red[i]);
  return t;
}

// Activation of the gate in a gated pair act(a w^T) * (a w2^T); a parameter of the products' epilogues, numbered in
// the order of the list in gates.def.
enum {
#define TQ_GATE(name, expr) TQ_GATE_##name,
#include "gates.def"
#undef TQ_GATE
  TQ_GATE_COUNT
};
__device__ __forceinline__ float gate_fn(float x, int kind) {
  switch (kind) {
#define TQ_GATE(name, expr) \
  case TQ_GATE_##name:      \
    return (expr);
#include "gates.def"
#undef TQ_GATE
  }
  return x;
}

// A gated pair with a limit (limit > 0): the gate's input is capped from above at the limit, the other factor is held
// within +-limit and raised by one, f(min(g, limit)) * (clamp(u, -limit, limit) + 1); limit 0: f(g) * u.
__device__ __forceinline__ float gated_pair(float g, float u, int kind, float limit) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit) + 1.0f;
  }
  return gate_fn(g, kind) * u;
}
// The limit that the products' launchers put into their argument blocks (tq_set_pair_limit sets it; 0: none).  It is
// read on the host when a launch is made and travels as a kernel argument from there on.
extern float tq_pair_limit_host;

#define TQ_LAUNCH_CHECK()                        \
  do {                                           \
    hipError_t e__ = hipGetLastError();          \
    if (e__ != hipSuccess) return (int)e__;      \
  } while (0)

// Calls `body` with `W` bound to the C type of a run-time weight type.
#define TQ_DISPATCH_W(wtype, ...)                  \
  do {                                             \
    if ((wtype) == TQ_F32) {                       \
      typedef float W;                             \
      __VA_ARGS__                                  \
    } else if ((wtype) == TQ_BF16) {               \
      typedef bf16_t W;                            \
      __VA_ARGS__                                  \
    } else {                                       \
      return TQ_ERR_BAD_ARG;                       \
    }                                              \
  } while (0)

#define TQ_API extern "C" __attribute__((visibility("default")))
