// Products of many rows in tiles of up to 256 x 256 outputs by two groups of four waves that take turns: while one group
// multiplies, the other reads its operands from LDS and asks for what comes later, and a barrier between the two phases
// lets them change places.  Same contract, operand layouts and order of sums as the tile kernel in gemm_mfma.hip: same bits.
//
// What bounds it: a tile of 64 of k is 64 KB on its way through L2 and 4.2 million multiply-adds, 0.85 us of the matrix
// instructions of a compute unit at their full clock and about as long as its path to L2 takes for the bytes, so each has to go on
// beside the other:
//  * a wave owns 32 MI x 64 outputs (MI up to 4), for which its reads from LDS (4 MI + 8 operand reads a tile of 64) take less time
//    than its products, and the group that multiplies has the matrix instructions to itself;
//  * loads go straight into LDS and are asked for by the reading group alone, behind its reads.  A wave that asks for more than the
//    path takes stands still until there is room, and in front of products or reads that time is lost: 13,197 tokens by 8 of 64
//    experts of 2,560 x 3,584 took 4,215 us with two loads in front of every phase of a wave and 3,739 this way;
//  * the tiles wait in rings of two (a) and three (w; four where an item has up to 128 rows) tiles, so that a tile of w is asked
//    for five to seven phases of 0.25 us before it is read: memory's time where an expert's matrices are read once.  Rings of half
//    tiles of 32 of k are level with two whole ones: rows of 64 bytes halve what L2 gives.
// One workgroup fills a compute unit's LDS, so what stands between two tiles has nothing to hide behind: the end of a workgroup and the
// start of the next (1.9 us on average, 5.8 for one in ten), the search for its tile (0.9), the first loads' way (3).  An order of rows has
// queues for that (PhaseTiles): a workgroup stays, and a die that is through helps the others: 2,048 tokens by 4 of 60 experts of 1,408 x
// 2,048 beside a shared one of 5,632 260 -> 244 us.  With w as the products'
// first operand a lane ends with columns side by side, and the outputs go from the registers into stores of 16 bytes a lane.  What is left
// of an end is the gate's arithmetic, 31 instructions a value as expf, a division and a rounding by integers make it, 9.5 us a tile of 256 x
// 128 beside 39 of its steps: 19 now (silu_within, f32_to_bf16), 244 -> 240 us there.
// What the matrix instructions cost is power: on random values the chip runs 32x32x16 products alone at 1,858 TFLOP/s and 16x16x32
// products at 2,183 (1.7 GHz in this kernel either way, where 2.4 is the peak), so these are the small ones.  They add k in groups of
// eight, one behind the other, as the large ones do: same bits.
// Measured, us, with items of two units by 16 waves through a ring of three stages, then these tiles by 32x32x16 products and outputs
// through LDS, then as it is: 13,197 tokens by 8 of 64 experts of 2,560 x 3,584 beside a shared expert of 20,480, gated pairs 7,551 ->
// 5,682 (1,363 TFLOP/s), second products 3,496 -> 3,041 (the experts alone 4,760 -> 3,739 and 2,590 -> 1,943 before); 2,048 tokens by 4
// of 60 experts of 1,408 x 2,048 beside one of 5,632 293 -> 240 and 165 -> 155 (the experts alone 219 -> 173 and 147 -> 103 before).
// Products of one matrix (`launch_gemm_phases_plain`) take the same tiles, 64 to 256 rows high as the compute units fill best; gemm_mfma.hip
// has the rules and what they replace (2,048 rows by 2,048 columns with a bias, k 2,048, 62 -> 27 us; 3,001 by 3,072 99 -> 43).
#include "common.h"

#include "gemm_mfma.h"

#define PH_FENCE()                        \
  do {                                    \
    asm volatile("" ::: "memory");        \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)
#define PH_NEXT()                         \
  do {                                    \
    PH_FENCE();                           \
    __builtin_amdgcn_s_barrier();         \
    PH_FENCE();                           \
  } while (0)
// s_waitcnt: vmcnt in bits 3..0 and 15..14, lgkmcnt in bits 11..8, expcnt in bits 6..4
#define PH_LDS_DONE() __builtin_amdgcn_s_waitcnt(0xC07F)
template <int N>
__device__ __forceinline__ void loads_left() {      // at most N loads of this wave are on their way
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// x / (1 + exp(-x)) of N values, none of them 87 or more in size, to the same bits as the general form (compared over all floats of that
// range), so that it makes no difference which form the other values of a wave ask for.  What is left out is what only the ends of the
// range need.  The exponential: reduction to a power of two (Cody and Waite), with log2(e) in two floats and the product's rounding error by
// a fused multiply-add.  The second float is the one that expf has here, whose neighbour is as near: with that one 15 results were the next
// float.  The quotient: a reciprocal that one Newton step sharpens, and one correction by the remainder, whose sign is changed so that -0
// stays -0.  17 instructions instead of 25.
template <int N>
__device__ __forceinline__ void silu_within(float (&v)[N]) {
#pragma clang fp contract(off)      // (p - n is to be of the rounded p, whose rest stands apart)
  constexpr float LOG2E = 1.44269504088896341f, LOG2E_REST = 0x1.4ae0bep-26f;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float x = v[j], p = -x * LOG2E, rest = fmaf(-x, LOG2E_REST, fmaf(-x, LOG2E, -p)), n = rintf(p);
    const float d = 1.0f + ldexpf(__builtin_amdgcn_exp2f((p - n) + rest), (int)n);
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    const float q = x * r;
    v[j] = fmaf(-fmaf(d, q, -x), r, q);
  }
}

// v[j] = f(v[j]), the switch once for all of them
template <int N>
__device__ __forceinline__ void gate_many(float (&v)[N], int kind) {
  if (kind == TQ_GATE_silu) {
    float far = 0.f;
#pragma unroll
    for (int j = 0; j < N; ++j) far = fmaxf(far, fabsf(v[j]));
    if (!__any(!(far < 87.f))) {
      silu_within(v);
      return;
    }
  }
  switch (kind) {
#define TQ_GATE(name, expr)                          \
  case TQ_GATE_##name:                               \
    _Pragma("unroll") for (int j = 0; j < N; ++j) {  \
      const float x = v[j];                          \
      v[j] = (expr);                                 \
    }                                                \
    break;
#include "gates.def"
#undef TQ_GATE
  }
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
// threadIdx.x as something the compiler knows nothing about, so that what follows from it is worked out again for every tile rather than
// kept in registers that the tile's sums and operands fill
__device__ __forceinline__ int thread_anew() {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  return tid;
}

struct No {
  static constexpr bool value = false;
};
struct Yes {
  static constexpr bool value = true;
};

// A tile as the loop over its steps sees it, and as its outputs do.
struct PhaseWork {
  const bf16_t *a_src[4], *w_src[4];      // where this thread's 16 bytes of a step's loads lie (see phase_begin)
  int units, steps;                       // units of 64 rows (1..4); steps of 64 of k
};
struct PhaseOut {
  void* out;
  int64_t ldc;
  const void* bias;
  int bias_type, N, gate, act1;
  float limit;
  int units, n0, n1, mw;                  // units; first column of either half of 128 (of a gated pair the same); this wave's first row
  unsigned long long live_lo, live_hi;    // which of its rows exist and are no padding
};

// What the place of a chunk of 16 bytes in row r of w's tile is turned by: sixteen lanes that read one chunk of the rows of a product's
// operand (16 neighbours, or four of every eight) find it in 16 places of 16 bytes of the 256 that the banks serve together.
template <bool OUT_ACT>
__device__ __forceinline__ int w_place(int r) { return OUT_ACT ? ((r >> 1) & 1) | ((r >> 3) & 3) << 1 : (r >> 1) & 7; }

// LDS: a [2 tiles][2 groups][one group's rows of a], then w [3 or 4 tiles][2 halves][128 columns], rows of 64 of k.
__device__ __forceinline__ int a_slot_of(int units) { return units * 32 * TBK; }
__device__ __forceinline__ int w_tiles_of(int units) { return units > 2 ? 3 : 4; }
#define PH_W_SLOT (128 * TBK)

__device__ __forceinline__ void ask_a(const PhaseWork& t, bf16_t* lds, int units, int wm, int wn, int step) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i < units) load_to_lds16(t.a_src[i] + step * TBK, lds + ((step & 1) * 2 + 1 - wm) * a_slot_of(units) + (i * 32 + wn * 8) * TBK);
}
__device__ __forceinline__ void ask_w(const PhaseWork& t, bf16_t* lds, int units, int wm, int wn, int step, int slot) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    load_to_lds16(t.w_src[i] + step * TBK, lds + 4 * a_slot_of(units) + (slot * 2 + wm) * PH_W_SLOT + (i * 32 + wn * 8) * TBK);
}

// The steps of a tile of 64 MI rows (32 MI of either group of waves), whose first loads are on their way (phase_begin); `fresh`: and
// nothing is behind them.  Sums: acc [rows 16 i ..][half][tile of its columns].  With a queue, wave 0 takes the number behind this tile
// from `ticket` some steps before the end.
template <int MI, bool OUT_ACT>
__device__ __forceinline__ void phase_steps(const PhaseWork& p, bf16_t* lds, bool fresh, int* ticket, int& taken, f32x4 (&acc)[2 * MI][2][2]) {
  constexpr int A_SLOT = MI * 32 * TBK, WT = MI > 2 ? 3 : 4;      // WT: tiles of w in LDS (of a: 2)
  bf16_t* As = lds;
  bf16_t* Ws = lds + 4 * A_SLOT;
  const int tid = thread_anew(), lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 4, wn = wave % 4;      // group; a wave's 32 columns of either half
  const int steps = p.steps;
  auto ask_a_of = [&](int t) { ask_a(p, lds, MI, wm, wn, t); };
  auto ask_w_of = [&](int t, int slot) { ask_w(p, lds, MI, wm, wn, t, slot); };

  // The products are v_mfma_f32_16x16x32_bf16 with w as the first operand: a lane's four sums are four columns of one row, D lane l =
  // row l % 16 of a, columns 4 (l / 16) + v of w.  Which of the wave's 32 columns of a half a tile's column i is, is free: where the
  // result is of 16 bits, 8 (i / 4) + 4 j + i % 4 for the half's tiles j = 0 and 1, so that a lane ends with eight columns side by side.
#pragma unroll
  for (int i = 0; i < 2 * MI; ++i)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int lr = lane % 16, lq = lane / 16, a_x = (lr >> 1) & 7;
  u32x4 af[2 * MI], wf[2][2];
  // 32 of k: half h of tile t, whose w lies in `slot`
  auto read = [&](int t, int slot, int h) {
    const bf16_t* A = As + ((t & 1) * 2 + wm) * A_SLOT + lr * TBK;
    const bf16_t* W = Ws + slot * 2 * PH_W_SLOT + wn * 32 * TBK;
    const int c = 4 * h + lq;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = OUT_ACT ? 8 * (lr / 4) + 4 * j + lr % 4 : 16 * j + lr;
        wf[b][j] = *reinterpret_cast<const u32x4*>(W + b * PH_W_SLOT + r * TBK + ((c ^ w_place<OUT_ACT>(r)) << 3));
      }
#pragma unroll
    for (int i = 0; i < 2 * MI; ++i) af[i] = *reinterpret_cast<const u32x4*>(A + i * 16 * TBK + ((c ^ a_x) << 3));
    PH_FENCE();
  };
  auto multiply = [&]() {
#pragma unroll
    for (int i = 0; i < 2 * MI; ++i)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[b][j]), __builtin_bit_cast(bf16x8, af[i]),
                                                                 acc[i][b][j], 0, 0, 0);
    PH_FENCE();
  };

  // Phases 4 t .. 4 t + 3 of group 0: read the first half of tile t, multiply it, read the second, multiply it; group 1 is one phase
  // behind.  What a phase asks for goes where every wave has read what lay there (a0, a1: the groups' rows of a; w0, w1: the halves
  // of w): phase 4 t a1 of t + 1, 4 t + 1 w1 and 4 t + 2 w0 of t + WT - 1 (in the place of tile t - 1's, last read in phase 4 t - 1),
  // 4 t + 3 a0 of t + 2 (in the place of tile t's, last read in phase 4 t + 2).  A wave waits for its own loads before the barrier
  // behind which another wave reads them: everything of tile t but a1 is read from phase 4 t on, a1 from 4 t + 1 on.
  if (!fresh) {      // behind the first loads stand stores, how many is not known: all of them
    loads_left<0>();
  } else if (wm == 0) {
    if (WT == 4) {
      if (steps > 2) loads_left<MI + 8>();
      else loads_left<MI>();
    } else if (steps > 1) loads_left<MI + 4>();
    else loads_left<MI>();
  } else {
    if (steps >= WT - 1) loads_left<4 * (WT - 2) + MI>();
    else loads_left<0>();
  }
  PH_NEXT();
  int slot = 0;      // of tile t's w; the slot of tile t + WT - 1 is the one before it
  auto before = [](int s) { return s ? s - 1 : WT - 1; };
  auto behind = [](int s) { return s + 1 < WT ? s + 1 : 0; };
  // `LAST`: the last tiles, behind which less is asked for
  auto first_group = [&](int t, auto last) {
    constexpr bool LAST = decltype(last)::value;
    read(t, slot, 0);
    if (!LAST || t + 1 < steps) ask_a_of(t + 1);
    // a1 of t has landed: behind it, the w0 asked for in phase 4 t - 2 and the a1 just asked for
    if (!LAST || t + WT - 2 < steps) loads_left<MI + 4>();
    else if (t + 1 < steps) loads_left<MI>();
    else loads_left<0>();
    PH_LDS_DONE();
    PH_NEXT();
    multiply();
    PH_NEXT();
    read(t, slot, 1);
    if (!LAST || t + WT - 1 < steps) ask_w_of(t + WT - 1, before(slot));
    PH_LDS_DONE();
    PH_NEXT();
    multiply();
    // w0 of t + 1 has landed
    if (!LAST || t + WT - 1 < steps) loads_left<(WT == 4 ? 8 : 4) + MI>();
    else if (WT == 4 && t + 2 < steps) loads_left<4 + MI>();
    else if (t + 1 < steps) loads_left<MI>();
    PH_NEXT();
    slot = behind(slot);
  };
  auto second_group = [&](int t, auto last) {
    constexpr bool LAST = decltype(last)::value;
    read(t, slot, 0);
    if (!LAST || t + WT - 1 < steps) ask_w_of(t + WT - 1, before(slot));
    PH_LDS_DONE();
    PH_NEXT();
    multiply();
    PH_NEXT();
    read(t, slot, 1);
    if (!LAST || t + 2 < steps) ask_a_of(t + 2);
    // a0 and w1 of t + 1 have landed: behind them, what this tile's phases asked for
    if (!LAST || t + WT - 1 < steps) loads_left<4 + MI>();
    else if (t + 2 < steps) loads_left<MI>();
    else loads_left<0>();
    PH_LDS_DONE();
    PH_NEXT();
    multiply();
    PH_NEXT();
    slot = behind(slot);
  };
  int t = 0;
  if (wm == 0) {
    for (; t + WT - 1 < steps; ++t) first_group(t, No());
    // (one more on its way only makes the waits behind it wait for one more)
    if (ticket && tid == 0) taken = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (; t < steps; ++t) first_group(t, Yes());
    PH_NEXT();      // phase 4 steps, in which group 1 multiplies
  } else {
    PH_NEXT();      // phase 0
    for (; t + WT - 1 < steps; ++t) second_group(t, No());
    for (; t < steps; ++t) second_group(t, Yes());
  }
}

// The outputs of a tile, 16 rows at a time, from the registers: a lane's pieces of 16 bytes, the four lanes of a row side by side.
template <int MI, bool DUAL, bool OUT_ACT>
__device__ __forceinline__ void phase_store(const PhaseOut& g, const f32x4 (&acc)[2 * MI][2][2]) {
  const int tid = thread_anew(), lane = tid % 64, wn = tid / 64 % 4, lr = lane % 16, lq = lane / 16;
  constexpr int V = OUT_ACT ? 8 : 4, HALVES = DUAL ? 1 : 2, J = OUT_ACT ? 1 : 2;      // columns of a piece; pieces of a lane's row
  const int col0 = wn * 32 + (OUT_ACT ? 8 : 4) * lq;
  float bias[HALVES][J][V];
#pragma unroll
  for (int b = 0; b < HALVES; ++b)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int n = (b ? g.n1 : g.n0) + col0 + 16 * j + v;
        bias[b][j][v] = g.bias && n < g.N ? g.bias_type == TQ_F32 ? ((const float*)g.bias)[n] : to_f32(((const bf16_t*)g.bias)[n]) : 0.f;
      }
  const bool aligned = g.ldc % V == 0 && (uintptr_t)g.out % 16 == 0;
  const bool even = g.N % 2 == 0 && g.ldc % 2 == 0 && (uintptr_t)g.out % 8 == 0;      // columns in pairs at least
#pragma unroll 1
  for (int i = 0; i < 2 * MI; ++i) {      // (kept a loop; the sums stay in registers since each case names its own)
    f32x4 sums[2][2];
// (each case's statement is its own, so that no two become one with the sums found by an address)
#define PH_TAKE(n)                                                                                                       \
  if constexpr (2 * MI > n)                                                                                              \
    if (i == n) {                                                                                                        \
      _Pragma("unroll") for (int b = 0; b < 2; ++b)                                                                      \
          _Pragma("unroll") for (int j = 0; j < 2; ++j) sums[b][j] = acc[n][b][j];                                       \
      asm volatile("" : "+v"(sums[0][0]), "+v"(sums[0][1]), "+v"(sums[1][0]), "+v"(sums[1][1]) : "n"(n));                \
    }
    PH_TAKE(0) PH_TAKE(1) PH_TAKE(2) PH_TAKE(3) PH_TAKE(4) PH_TAKE(5) PH_TAKE(6) PH_TAKE(7)
#undef PH_TAKE
    if (!(((i < 4 ? g.live_lo : g.live_hi) >> (i % 4 * 16 + lr)) & 1)) continue;
    const size_t row = (size_t)(g.mw + 16 * i + lr) * g.ldc;
#pragma unroll
    for (int b = 0; b < HALVES; ++b)
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int col = (b ? g.n1 : g.n0) + col0 + 16 * j;
        float v[V];
#pragma unroll
        for (int k = 0; k < V; ++k) v[k] = sums[b][OUT_ACT ? k / 4 : j][k % 4] + bias[b][j][k];
        if (DUAL) {
          float u[V];
#pragma unroll
          for (int k = 0; k < V; ++k) u[k] = sums[1][OUT_ACT ? k / 4 : j][k % 4];
          if (g.limit > 0.f) {
#pragma unroll
            for (int k = 0; k < V; ++k) {
              v[k] = fminf(v[k], g.limit);
              u[k] = fminf(fmaxf(u[k], -g.limit), g.limit) + 1.0f;
            }
          }
          gate_many(v, g.gate);
#pragma unroll
          for (int k = 0; k < V; ++k) v[k] *= u[k];
        } else if (g.act1) {
          gate_many(v, g.act1 - 1);
        }
        const bool wide = aligned && col + V <= g.N;
        if constexpr (OUT_ACT) {
          bf16_t* o = (bf16_t*)g.out + row + col;
          if (wide) {
            u32x4 packed;
#pragma unroll
            for (int k = 0; k < 4; ++k) packed[k] = f32_to_bf16_pair(v[2 * k], v[2 * k + 1]);
            *reinterpret_cast<u32x4*>(o) = packed;
          } else if (even) {
#pragma unroll
            for (int k = 0; k < V; k += 2)
              if (col + k < g.N) *reinterpret_cast<unsigned*>(o + k) = f32_to_bf16_pair(v[k], v[k + 1]);
          } else {
#pragma unroll
            for (int k = 0; k < V; ++k)
              if (col + k < g.N) o[k] = f32_to_bf16(v[k]);
          }
        } else {
          float* o = (float*)g.out + row + col;
          if (wide) {
            *reinterpret_cast<f32x4*>(o) = f32x4{v[0], v[1], v[2], v[3]};
          } else if (even) {
#pragma unroll
            for (int k = 0; k < V; k += 2)
              if (col + k < g.N) *reinterpret_cast<f32x2*>(o + k) = f32x2{v[k], v[k + 1]};
          } else {
#pragma unroll
            for (int k = 0; k < V; ++k)
              if (col + k < g.N) o[k] = v[k];
          }
        }
      }
  }
}

// Where tile `logical` of a product lies, in the order in which a die goes through its run of them, and its first loads.  A matrix per
// expert (the first product): expert by expert, so that an expert's matrices are read by one die, and within an expert column by column
// with its items side by side.  One matrix (the second): tiles of `rows` rows in bands of 8, down a band's columns, a run of k behind
// the other.
template <bool DUAL, bool OUT_ACT>
__device__ __forceinline__ void phase_begin(MfmaGemmArgs g, int logical, int gx, int gy, int n_units, int rows, bf16_t* lds, PhaseWork& t, PhaseOut& o) {
  const int tid = thread_anew(), lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 4, wn = wave % 4;
  int tile_n, group = 0, m0, units;
  if (g.tile_group) {
    const int* items = g.tile_group + g.M / 64;
    const int n_items = gx, at = logical / gy;
    // The expert's items lo .. hi - 1: among the 64 around this one, unless they reach beyond those.
    const int first = max(at - 31, 0), c = min(first + lane, n_items - 1);
    const int unit = items[c], expert = g.tile_group[unit];
    group = __builtin_amdgcn_readlane(expert, at - first);
    const unsigned long long same = __ballot(expert == group && first + lane < n_items);
    const int here = at - first;
    const unsigned long long others_below = ~same & ((1ull << here) - 1ull), others_above = ~same >> here;      // (bit 0: this one, clear)
    int lo = others_below ? first + 64 - __builtin_clzll(others_below) : first;
    int hi = others_above ? at + __builtin_ctzll(others_above) : first + 64;
    for (bool more = !others_below && first > 0; more;) {
      const int b = lo - 1 - lane;
      const unsigned long long as = __ballot(b >= 0 && g.tile_group[items[max(b, 0)]] == group);
      lo -= ~as ? __builtin_ctzll(~as) : 64;
      more = !~as;
    }
    for (bool more = !others_above; more;) {
      const int b = hi + lane;
      const unsigned long long as = __ballot(b < n_items && g.tile_group[items[min(b, n_items - 1)]] == group);
      hi += ~as ? __builtin_ctzll(~as) : 64;
      more = !~as;
    }
    const int local = logical - lo * gy, n_e = hi - lo;
    tile_n = local / n_e;
    const int item = lo + local % n_e, place = item - first;
    const bool near = place >= 0 && place + 1 < 64;
    const int u0 = near ? __builtin_amdgcn_readlane(unit, place & 63) : items[item];
    const int next = item + 1 >= n_items ? n_units : near ? __builtin_amdgcn_readlane(unit, (place + 1) & 63) : items[item + 1];
    m0 = u0 * 64;
    units = min(next - u0, 4);
  } else {
    const int run = logical / (gx * gy);
    logical %= gx * gy;
    if (g.k_per < g.K) {      // partial sums: run z of k, its sums to out + z * split_stride, the bias with run 0
      const int k_lo = run * g.k_per;
      g.a += k_lo;
      g.w += k_lo;
      g.out = (float*)g.out + run * g.split_stride;
      if (run) g.bias = nullptr;
      g.k_per = min(g.k_per, g.K - k_lo);
    }
    const int band = logical / (8 * gy), in_band = logical % (8 * gy), bh = min(8, gx - band * 8);
    tile_n = in_band / bh;
    m0 = (band * 8 + in_band % bh) * rows;
    units = min((g.M - m0 + 63) / 64, rows / 64);
  }
  units = __builtin_amdgcn_readfirstlane(units);
  m0 = __builtin_amdgcn_readfirstlane(m0);
  const bf16_t* w = (DUAL && wm ? g.w2 : g.w) + (size_t)group * g.group_stride;
  const int n0 = tile_n * (DUAL ? 128 : 256), n1 = DUAL ? n0 : n0 + 128;
  t.units = units;
  t.steps = g.k_per / TBK;
  // What this thread asks for: group 0 the rows of a that group 1 multiplies and the first half of w, group 1 the others; rows
  // row + 32 i, the chunk of 16 bytes that belongs at place tid % 8 (the swizzle is in what is asked for).  Rows past the end
  // and rows of padding read some valid row instead: those outputs are never stored.
  const int row = (tid % 256) / 8, chunk = (tid % 8) ^ ((row >> 1) & 7), w_chunk = (tid % 8) ^ w_place<OUT_ACT>(row);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = min(m0 + (1 - wm) * 32 * units + row + 32 * i, g.M - 1);
    int src = m;
    if (g.a_rows && g.a_gather) src = max(g.a_rows[m], 0);
    t.a_src[i] = g.a + (size_t)src * g.lda + chunk * 8;
    t.w_src[i] = w + (size_t)min((wm ? n1 : n0) + row + 32 * i, g.N - 1) * g.K + w_chunk * 8;
  }
  // which of this wave's rows exist and are no padding (for the stores; asked for here, where nothing waits behind them)
  const int mw = m0 + wm * 32 * units;
  auto alive = [&](int r) { return __ballot(r < 32 * units && mw + r < g.M && !(g.a_rows && g.a_rows[min(mw + r, g.M - 1)] < 0)); };
  o = PhaseOut{g.out, g.ldc, g.bias, g.bias_type, g.N, g.gate, g.act1, g.limit, units, n0, n1, mw, alive(lane), alive(64 + lane)};
  PH_FENCE();
  const int wt = w_tiles_of(units);
  if (wm == 0) {
    ask_w(t, lds, units, wm, wn, 0, 0);
    if (wt == 4 && t.steps > 1) ask_w(t, lds, units, wm, wn, 1, 1);
    ask_a(t, lds, units, wm, wn, 0);
    if (wt == 4 ? t.steps > 2 : t.steps > 1) ask_w(t, lds, units, wm, wn, wt - 2, wt - 2);
  } else {
    ask_a(t, lds, units, wm, wn, 0);
    ask_w(t, lds, units, wm, wn, 0, 0);
    for (int s = 1; s < wt - 1; ++s)
      if (s < t.steps) ask_w(t, lds, units, wm, wn, s, s);
    if (t.steps > 1) ask_a(t, lds, units, wm, wn, 1);
  }
  PH_FENCE();
}

// The tiles of a launch: a die (workgroups are dealt to the 8 of them in turn) gets a contiguous run of those of the first product and one
// of the second's, if there is one (n2 tiles of `rows2` rows, gx2 x gy2 a run of k): `first2`: the second's before the first's, else spread
// among them.  A first without an order of rows is not there at all: the second alone.
// queue (or null: a workgroup has one tile, that of its number): eight numbers, zero before the launch, one a die: a workgroup takes the
// next tile of its die's run until there is none, then of that with most left, and the loads of a tile's first steps are on their way
// while the outputs of the one before are stored.
struct PhaseTiles {
  int gx, gy, n_units, gx2, gy2, rows2, first2, q1, rem1, q2, rem2;
  int* queue;
  __device__ __forceinline__ int first(int die) const { return q1 + (die < rem1 ? 1 : 0); }
  __device__ __forceinline__ int second(int die) const { return q2 + (die < rem2 ? 1 : 0); }
  __device__ __forceinline__ int of(int die) const { return first(die) + second(die); }
};

// The tile behind `taken`, the number that wave 0's first lane has from its die's queue (and has to take first if `fresh`), for all waves,
// none of which is still reading LDS; false: there is none.
__device__ __forceinline__ bool phase_next(const PhaseTiles& s, bool fresh, int taken, int* word, int& die, int& i) {
  const int tid = thread_anew(), lane = tid % 64;
  if (__builtin_amdgcn_readfirstlane(tid / 64) == 0) {
    if (fresh && lane == 0) taken = __hip_atomic_fetch_add(s.queue + die, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    i = __builtin_amdgcn_readfirstlane(taken);
    while (die >= 0 && i >= s.of(die)) {      // (a die that was tried in vain has nothing left from then on: at most eight times)
      const int left = s.of(lane % 8) - __hip_atomic_load(s.queue + lane % 8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int most = 0;
      die = -1;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const int l = __builtin_amdgcn_readlane(left, d);
        if (l > most) most = l, die = d;
      }
      if (die < 0) break;
      if (lane == 0) taken = __hip_atomic_fetch_add(s.queue + die, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      i = __builtin_amdgcn_readfirstlane(taken);
    }
    if (lane == 0) word[0] = die, word[1] = i;      // LDS's first words carry the answer
  }
  __syncthreads();
  die = __builtin_amdgcn_readfirstlane(word[0]);
  i = __builtin_amdgcn_readfirstlane(word[1]);
  __syncthreads();
  return die >= 0;
}

template <bool DUAL, bool OUT_ACT>
__device__ __forceinline__ void phase_begin_of(const PhaseTiles& s, const MfmaGemmArgs& g, const MfmaGemmArgs& g2, int die, int i, bf16_t* lds,
                                               PhaseWork& work, PhaseOut& out) {
  const int mine1 = s.first(die), mine2 = s.second(die);
  int in2;      // how many of the second's tiles stand before this place
  bool second;
  if (s.first2) {
    in2 = min(i, mine2);
    second = i < mine2;
  } else {
    in2 = (int)((int64_t)i * mine2 / (mine1 + mine2));
    second = (int)((int64_t)(i + 1) * mine2 / (mine1 + mine2)) > in2;
  }
  const int logical = second ? die * s.q2 + min(die, s.rem2) + in2 : die * s.q1 + min(die, s.rem1) + i - in2;
  phase_begin<DUAL, OUT_ACT>(second ? g2 : g, logical, second ? s.gx2 : s.gx, second ? s.gy2 : s.gy, s.n_units, s.rows2, lds, work, out);
}

// One tile, and the beginning of the next if there is one.
template <int MI, bool DUAL, bool OUT_ACT>
__device__ __forceinline__ bool phase_tile(const PhaseTiles& s, const MfmaGemmArgs& g, const MfmaGemmArgs& g2, bool fresh, int& die, bf16_t* lds,
                                           PhaseWork& work, PhaseOut& out) {
  f32x4 acc[2 * MI][2][2];
  int taken = 0, i = 0;
  phase_steps<MI, OUT_ACT>(work, lds, fresh, s.queue ? s.queue + die : nullptr, taken, acc);
  const PhaseOut done = out;
  const bool more = s.queue && phase_next(s, false, taken, (int*)lds, die, i);
  if (more) phase_begin_of<DUAL, OUT_ACT>(s, g, g2, die, i, lds, work, out);
  phase_store<MI, DUAL, OUT_ACT>(done, acc);
  return more;
}

template <bool DUAL, bool OUT_ACT>
__global__ __launch_bounds__(512) void gemm_phases_kernel(MfmaGemmArgs g, int gy, MfmaGemmArgs g2, int gx2, int gy2, int n2, int rows2, int first2,
                                                          int* queue) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* lds = (bf16_t*)smem;
  PhaseTiles s;
  s.n_units = g.tile_group ? min(g.n_tiles[0], g.M / 64) : 0;
  s.gx = g.tile_group ? min(g.n_tiles[1], g.M / 64) : 0;
  s.gy = gy, s.gx2 = gx2, s.gy2 = gy2, s.rows2 = rows2, s.first2 = first2, s.queue = queue;
  const int n1 = s.gx * gy;
  if (queue) {
    // Where the experts' matrices pass for many rows each, or for so few that nothing else counts, the second's tiles go first, all of
    // them reading what their dies' L2 holds; between, where memory and the matrix instructions are about in balance (1,280 TFLOP/s
    // against 5.5 TB/s: 230 rows), they are spread among those that wait for memory.  us spread and first, gated pairs of 60 experts of
    // 1,408 x 2,048 beside one of 5,632: 60 rows each 191 and 179, 100 203 and 222, 137 241 and 253, 200 275 and 296, 260 361 and 369,
    // 330 456 and 445, 1,650 1,848 and 1,795; 64 of 2,560 x 3,584 beside 20,480: 60 543 and 547, 137 713 and 751, 260 1,170 and 1,121,
    // 1,650 6,190 and 5,688.  (With padding 260 rows are 291 of the 60 and 290 of the 64: the upper line lies where the narrower experts lose
    // 2 % and the wider gain 4, and between 200 and 260 nothing was timed.)
    const int per_expert = s.n_units * 64 / max(g.n_tiles[2], 1);      // rows, padding among them
    if (per_expert >= 270 || per_expert <= 100) s.first2 = 1;
  }
  s.q1 = n1 / 8, s.rem1 = n1 % 8, s.q2 = n2 / 8, s.rem2 = n2 % 8;
  int die = blockIdx.x % 8, i = blockIdx.x / 8;
  if (queue) {
    if (!phase_next(s, true, 0, (int*)smem, die, i)) return;
  } else if (i >= s.of(die)) {
    return;
  }
  PhaseWork work;
  PhaseOut out;
  phase_begin_of<DUAL, OUT_ACT>(s, g, g2, die, i, lds, work, out);
  bool more = true;
  for (bool fresh = true; more; fresh = false) switch (work.units) {
      case 4: more = phase_tile<4, DUAL, OUT_ACT>(s, g, g2, fresh, die, lds, work, out); break;
      case 3: more = phase_tile<3, DUAL, OUT_ACT>(s, g, g2, fresh, die, lds, work, out); break;
      case 2: more = phase_tile<2, DUAL, OUT_ACT>(s, g, g2, fresh, die, lds, work, out); break;
      default: more = phase_tile<1, DUAL, OUT_ACT>(s, g, g2, fresh, die, lds, work, out);
    }
}

static int launch_phases(const MfmaGemmArgs& g, int gy, int64_t n1, const MfmaGemmArgs& g2, int gx2, int gy2, int64_t n2, int rows2, int first2,
                         int* queue, bool dual, bool out_act, hipStream_t st) {
  int64_t per_die = (n1 + 7) / 8 + (n2 + 7) / 8;
  if (per_die * 8 > 0x7fffffff) return TQ_ERR_UNSUPPORTED;
  if (queue && per_die > 32) per_die = 32;      // a workgroup for each of the 256 compute units
  const int shmem = 160 * 1024;      // MI = 2 and 4; 144 KB where MI is 1 or 3
#define TQ_PHASES(D, O)                                                                                                       \
  do {                                                                                                                        \
    if (hipFuncSetAttribute((const void*)gemm_phases_kernel<D, O>, hipFuncAttributeMaxDynamicSharedMemorySize, shmem) != hipSuccess) \
      return TQ_ERR_UNSUPPORTED;                                                                                              \
    hipLaunchKernelGGL((gemm_phases_kernel<D, O>), dim3((unsigned)(per_die * 8)), dim3(512), shmem, st, g, gy, g2, gx2, gy2,  \
                       (int)n2, rows2, first2, queue);                                                                        \
  } while (0)
  if (dual && out_act) TQ_PHASES(true, true);
  else if (dual) TQ_PHASES(true, false);
  else if (out_act) TQ_PHASES(false, true);
  else TQ_PHASES(false, false);
#undef TQ_PHASES
  return 0;
}

// g2 (null: none): a second product, of one matrix and of the same kind, whose tiles fill the chip beside the first's; its k may be
// in runs (k_per, split_stride).  queue (or null): as for the kernel.
int launch_gemm_phases(const MfmaGemmArgs& g, const MfmaGemmArgs* g2, int* queue, bool dual, bool out_act, hipStream_t st) {
  if (!g.tile_group || !g.n_tiles) return TQ_ERR_BAD_ARG;
  const int cols = dual ? 128 : 256;
  const int gx = g.M / 64, gy = (g.N + cols - 1) / cols;      // (units of 64 rows: at most so many items)
  int gx2 = 1, gy2 = 1, n2 = 0, first2 = 0;
  if (g2) {
    gx2 = (g2->M + 255) / 256, gy2 = (g2->N + cols - 1) / cols;
    n2 = gx2 * gy2 * ((g2->K + g2->k_per - 1) / g2->k_per);
    // Tiles that take longer start first.  60 experts of 2,048 x 1,408, us with the second's tiles first and spread among the first's:
    // 2,048 rows beside runs of 2,816 of k 143 and 164, beside 1,024 x 2,048 of 2,048 107 and 126, 13,197 rows of 5,632 613 and 706.
    // Tiles of about the same time gain less: 2,048 rows of k 1,920 131 and 144, of 1,408 136 and 139, of 704 130 and 130; 1,100 rows
    // in runs of 1,408 120 and 131; 6,000 rows of 1,408 to 2,112 level (and vary by 4 %); gated pairs beside 1,408 columns 195 and 204,
    // beside 5,632 261 and 266.  No side where spreading wins was found: the line is no border between two, only where the gain is sure.
    first2 = g2->k_per >= 3 * g.K / 2;
  }
  return launch_phases(g, gy, (int64_t)gx * gy, g2 ? *g2 : g, gx2, gy2, n2, 256, first2, queue, dual, out_act, st);
}

// A product of one matrix, whose rows follow one another, in tiles of `rows` (a multiple of 64 up to 256) rows; k may be in runs.
int launch_gemm_phases_plain(const MfmaGemmArgs& g, int rows, bool dual, bool out_act, hipStream_t st) {
  if (g.tile_group || g.a_rows) return TQ_ERR_BAD_ARG;
  const int cols = dual ? 128 : 256;
  const int64_t gx = (g.M + rows - 1) / rows, gy = (g.N + cols - 1) / cols, n = gx * gy * ((g.K + g.k_per - 1) / g.k_per);
  if (n > (1 << 28)) return TQ_ERR_UNSUPPORTED;
  return launch_phases(g, 1, 0, g, (int)gx, (int)gy, n, rows, 0, nullptr, dual, out_act, st);
}

// Into how many runs the second product's k goes beside a first of M1 rows (at most): so many that none of its tiles takes longer than
// the chip has to do for both, while a run keeps 1,024 of k and the partial sums, which the kernel behind reads, stay within 256 MB.
TQ_API int tq_gemm_phases_pair_splits(int M1, int N1, int K1, int M2, int N2, int K2) {
  const int64_t tiles1 = (int64_t)(M1 + 255) / 256 * ((N1 + 255) / 256), tiles2 = (int64_t)(M2 + 255) / 256 * ((N2 + 255) / 256);
  const int64_t all = (tiles1 * K1 + tiles2 * K2) / 256;
  int s = 1;
  while (s < 8 && K2 / s > all && K2 / (2 * s) >= 1024 && (int64_t)2 * s * M2 * N2 * 4 <= (256 << 20)) s *= 2;
  while (s > 1 && (int64_t)(s - 1) * (((K2 + TBK - 1) / TBK + s - 1) / s * TBK) >= K2) s /= 2;      // every run begins before the end of k
  return s;
}
