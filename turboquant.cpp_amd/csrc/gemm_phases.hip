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
// One workgroup fills a compute unit's LDS, so what the waves do behind the last tile has nothing to hide behind: with w as the products'
// first operand a lane ends with columns side by side, and the outputs go from the registers into stores of 16 bytes a lane.
// What the matrix instructions cost is power: on random values the chip runs 32x32x16 products alone at 1,858 TFLOP/s and 16x16x32
// products at 2,183 (1.7 GHz in this kernel either way, where 2.4 is the peak), so these are the small ones.  They add k in groups of
// eight, one behind the other, as the large ones do: same bits.
// Measured, us, with items of two units by 16 waves through a ring of three stages, then these tiles by 32x32x16 products and outputs
// through LDS, then as it is: 13,197 tokens by 8 of 64 experts of 2,560 x 3,584 beside a shared expert of 20,480, gated pairs 7,551 ->
// 6,334 (1,223 TFLOP/s), second products 3,496 -> 3,051 (the experts alone 4,760 -> 3,739 and 2,590 -> 1,943 before); 2,048 tokens by 4
// of 60 experts of 1,408 x 2,048 beside one of 5,632 293 -> 260 and 165 -> 154 (the experts alone 219 -> 173 and 147 -> 103 before).
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

// v[j] = f(v[j]), the switch once for all of them
template <int N>
__device__ __forceinline__ void gate_many(float (&v)[N], int kind) {
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
struct No {
  static constexpr bool value = false;
};
struct Yes {
  static constexpr bool value = true;
};

struct PhaseTile {
  int m0, units;               // first row and units of 64 rows (1..4)
  int n0, n1;                  // first column of either half of 128 columns (the other matrix's same columns for a gated pair)
  const bf16_t *w, *w2;        // the matrices of the halves
};

// What the place of a chunk of 16 bytes in row r of w's tile is turned by: sixteen lanes that read one chunk of the rows of a product's
// operand (16 neighbours, or four of every eight) find it in 16 places of 16 bytes of the 256 that the banks serve together.
template <bool OUT_ACT>
__device__ __forceinline__ int w_place(int r) { return OUT_ACT ? ((r >> 1) & 1) | ((r >> 3) & 3) << 1 : (r >> 1) & 7; }

// One tile of 64 MI rows (32 MI of either group of waves).
template <int MI, bool DUAL, bool OUT_ACT>
__device__ __forceinline__ void phases_tile(const MfmaGemmArgs& g, const PhaseTile& p, bf16_t* lds) {
  constexpr int A_SLOT = MI * 32 * TBK, W_SLOT = 128 * TBK;      // one group's rows of a, one half of w
  constexpr int WT = MI > 2 ? 3 : 4;                             // tiles of w in LDS (of a: 2)
  bf16_t* As = lds;                                              // [2 tiles][2 groups][A_SLOT]
  bf16_t* Ws = lds + 4 * A_SLOT;                                 // [WT tiles][2 halves][W_SLOT]
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 4, wn = wave % 4;      // group; a wave's 32 columns of either half
  const int steps = g.k_per / TBK;

  // What this thread asks for: group 0 the rows of a that group 1 multiplies and the first half of w, group 1 the others; rows
  // row + 32 i, the chunk of 16 bytes that belongs at place tid % 8 (the swizzle is in what is asked for).  Rows past the end
  // and rows of padding read some valid row instead: those outputs are never stored.
  const int row = (tid % 256) / 8, chunk = (tid % 8) ^ ((row >> 1) & 7), w_chunk = (tid % 8) ^ w_place<OUT_ACT>(row);
  const bf16_t *a_src[MI], *w_src[4];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = min(p.m0 + (1 - wm) * 32 * MI + row + 32 * i, g.M - 1);
    int src = m;
    if (g.a_rows && g.a_gather) src = max(g.a_rows[m], 0);
    a_src[i] = g.a + (size_t)src * g.lda + chunk * 8;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) w_src[i] = (wm ? p.w2 : p.w) + (size_t)min((wm ? p.n1 : p.n0) + row + 32 * i, g.N - 1) * g.K + w_chunk * 8;
  auto ask_a = [&](int t) {
#pragma unroll
    for (int i = 0; i < MI; ++i) load_to_lds16(a_src[i] + t * TBK, As + ((t & 1) * 2 + 1 - wm) * A_SLOT + (i * 32 + wn * 8) * TBK);
  };
  auto ask_w = [&](int t, int slot) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds16(w_src[i] + t * TBK, Ws + (slot * 2 + wm) * W_SLOT + (i * 32 + wn * 8) * TBK);
  };

  // which of this wave's rows exist and are no padding (the epilogue's stores; asked for here, where nothing waits behind them)
  const int mw = p.m0 + wm * 32 * MI;
  auto alive = [&](int r) { return __ballot(r < 32 * MI && mw + r < g.M && !(g.a_rows && g.a_rows[min(mw + r, g.M - 1)] < 0)); };
  const unsigned long long live_lo = alive(lane), live_hi = MI > 2 ? alive(64 + lane) : 0;

  // The products are v_mfma_f32_16x16x32_bf16 with w as the first operand: a lane's four sums are four columns of one row, D lane l =
  // row l % 16 of a, columns 4 (l / 16) + v of w.  Which of the wave's 32 columns of a half a tile's column i is, is free: where the
  // result is of 16 bits, 8 (i / 4) + 4 j + i % 4 for the half's tiles j = 0 and 1, so that a lane ends with eight columns side by side.
  f32x4 acc[2 * MI][2][2];      // [rows 16 i ..][half][tile of its columns]
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
    const bf16_t* W = Ws + slot * 2 * W_SLOT + wn * 32 * TBK;
    const int c = 4 * h + lq;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = OUT_ACT ? 8 * (lr / 4) + 4 * j + lr % 4 : 16 * j + lr;
        wf[b][j] = *reinterpret_cast<const u32x4*>(W + b * W_SLOT + r * TBK + ((c ^ w_place<OUT_ACT>(r)) << 3));
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
  if (wm == 0) {
    ask_w(0, 0);
    if (WT == 4 && steps > 1) ask_w(1, 1);
    ask_a(0);
    if (WT == 4 ? steps > 2 : steps > 1) ask_w(WT - 2, WT - 2);
    if (WT == 4) {
      if (steps > 2) loads_left<MI + 8>();
      else loads_left<MI>();
    } else if (steps > 1) loads_left<MI + 4>();
    else loads_left<MI>();
  } else {
    ask_a(0);
    ask_w(0, 0);
#pragma unroll
    for (int t = 1; t < WT - 1; ++t)
      if (t < steps) ask_w(t, t);
    if (steps > 1) ask_a(1);
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
    if (!LAST || t + 1 < steps) ask_a(t + 1);
    // a1 of t has landed: behind it, the w0 asked for in phase 4 t - 2 and the a1 just asked for
    if (!LAST || t + WT - 2 < steps) loads_left<MI + 4>();
    else if (t + 1 < steps) loads_left<MI>();
    else loads_left<0>();
    PH_LDS_DONE();
    PH_NEXT();
    multiply();
    PH_NEXT();
    read(t, slot, 1);
    if (!LAST || t + WT - 1 < steps) ask_w(t + WT - 1, before(slot));
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
    if (!LAST || t + WT - 1 < steps) ask_w(t + WT - 1, before(slot));
    PH_LDS_DONE();
    PH_NEXT();
    multiply();
    PH_NEXT();
    read(t, slot, 1);
    if (!LAST || t + 2 < steps) ask_a(t + 2);
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
    for (; t < steps; ++t) first_group(t, Yes());
    PH_NEXT();      // phase 4 steps, in which group 1 multiplies
  } else {
    PH_NEXT();      // phase 0
    for (; t + WT - 1 < steps; ++t) second_group(t, No());
    for (; t < steps; ++t) second_group(t, Yes());
  }

  // The outputs, 16 rows at a time, from the registers: a lane's pieces of 16 bytes, the four lanes of a row side by side.
  constexpr int V = OUT_ACT ? 8 : 4, HALVES = DUAL ? 1 : 2, J = OUT_ACT ? 1 : 2;      // columns of a piece; pieces of a lane's row
  const int col0 = wn * 32 + (OUT_ACT ? 8 : 4) * lq;
  float bias[HALVES][J][V];
#pragma unroll
  for (int b = 0; b < HALVES; ++b)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int n = (b ? p.n1 : p.n0) + col0 + 16 * j + v;
        bias[b][j][v] = n < g.N ? bias_at(g, n) : 0.f;
      }
  const bool aligned = g.ldc % V == 0 && (uintptr_t)g.out % 16 == 0;
  const bool even = g.N % 2 == 0 && g.ldc % 2 == 0 && (uintptr_t)g.out % 8 == 0;      // columns in pairs at least
#pragma unroll 1
  for (int i = 0; i < 2 * MI; ++i) {      // (kept a loop; the sums stay in registers since each case names its own)
    f32x4 sums[2][2];
#define PH_TAKE(n)                                                        \
  if constexpr (2 * MI > n)                                               \
    if (i == n) {                                                         \
      _Pragma("unroll") for (int b = 0; b < 2; ++b)                       \
          _Pragma("unroll") for (int j = 0; j < 2; ++j) sums[b][j] = acc[n][b][j]; \
    }
    PH_TAKE(0) PH_TAKE(1) PH_TAKE(2) PH_TAKE(3) PH_TAKE(4) PH_TAKE(5) PH_TAKE(6) PH_TAKE(7)
#undef PH_TAKE
    if (!(((i < 4 ? live_lo : live_hi) >> (i % 4 * 16 + lr)) & 1)) continue;
    const size_t row = (size_t)(mw + 16 * i + lr) * g.ldc;
#pragma unroll
    for (int b = 0; b < HALVES; ++b)
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int col = (b ? p.n1 : p.n0) + col0 + 16 * j;
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
            for (int k = 0; k < 4; ++k) packed[k] = f32_to_bf16(v[2 * k]).bits | (unsigned)f32_to_bf16(v[2 * k + 1]).bits << 16;
            *reinterpret_cast<u32x4*>(o) = packed;
          } else if (even) {
#pragma unroll
            for (int k = 0; k < V; k += 2)
              if (col + k < g.N) *reinterpret_cast<unsigned*>(o + k) = f32_to_bf16(v[k]).bits | (unsigned)f32_to_bf16(v[k + 1]).bits << 16;
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

// Tile `logical` of a product in the order in which a die goes through its run of them.  A matrix per expert (the first product): expert
// by expert, so that an expert's matrices are read by one die, and within an expert column by column with its items side by side.
// One matrix (the second): tiles of `rows` rows in bands of 8, down a band's columns, a run of k behind the other.
template <bool DUAL>
__device__ __forceinline__ void phase_tile_of(MfmaGemmArgs& g, int logical, int gx, int gy, int rows, PhaseTile& p) {
  const int lane = threadIdx.x % 64;
  int tile_n, group = 0;
  if (g.tile_group) {
    const int units_all = g.M / 64;
    const int* items = g.tile_group + units_all;
    const int n_units = min(g.n_tiles[0], units_all), n_items = gx;
    const int at = logical / gy;
    group = g.tile_group[items[at]];
    // the expert's items lo .. hi - 1, 64 candidates at a time
    int lo = at, hi = at + 1;
    for (bool more = true; more;) {
      const int c = lo - 1 - lane;
      const unsigned long long same = __ballot(c >= 0 && g.tile_group[items[max(c, 0)]] == group);
      lo -= ~same ? __builtin_ctzll(~same) : 64;
      more = !~same;
    }
    for (bool more = true; more;) {
      const int c = hi + lane;
      const unsigned long long same = __ballot(c < n_items && g.tile_group[items[min(c, n_items - 1)]] == group);
      hi += ~same ? __builtin_ctzll(~same) : 64;
      more = !~same;
    }
    const int local = logical - lo * gy, n_e = hi - lo;
    tile_n = local / n_e;
    const int item = lo + local % n_e, u0 = items[item];
    p.m0 = u0 * 64;
    p.units = min((item + 1 < n_items ? items[item + 1] : n_units) - u0, 4);
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
    p.m0 = (band * 8 + in_band % bh) * rows;
    p.units = min((g.M - p.m0 + 63) / 64, rows / 64);
  }
  p.w = g.w + (size_t)group * g.group_stride;
  p.w2 = DUAL ? g.w2 + (size_t)group * g.group_stride : p.w;
  p.n0 = tile_n * (DUAL ? 128 : 256);
  p.n1 = DUAL ? p.n0 : p.n0 + 128;
}
template <bool DUAL, bool OUT_ACT>
__device__ __forceinline__ void phases(MfmaGemmArgs& g, int logical, int gx, int gy, int rows, bf16_t* lds) {
  PhaseTile p;
  phase_tile_of<DUAL>(g, logical, gx, gy, rows, p);
  switch (__builtin_amdgcn_readfirstlane(p.units)) {
    case 4: phases_tile<4, DUAL, OUT_ACT>(g, p, lds); break;
    case 3: phases_tile<3, DUAL, OUT_ACT>(g, p, lds); break;
    case 2: phases_tile<2, DUAL, OUT_ACT>(g, p, lds); break;
    default: phases_tile<1, DUAL, OUT_ACT>(g, p, lds);
  }
}

// A die (workgroups are dealt to the 8 of them in turn) gets a contiguous run of the tiles of the first product and one of the
// second, if there is one (n2 tiles of `rows2` rows, gx2 x gy2 a run of k): `first2`: the second's before the first's, else spread
// among them.  A first without an order of rows is not there at all: the second alone.
template <bool DUAL, bool OUT_ACT>
__global__ __launch_bounds__(512) void gemm_phases_kernel(MfmaGemmArgs g, int gy, MfmaGemmArgs g2, int gx2, int gy2, int n2, int rows2, int first2) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int gx = g.tile_group ? min(g.n_tiles[1], g.M / 64) : 0;
  const int id = blockIdx.x, die = id % 8, i = id / 8;
  const int n1 = gx * gy;
  const int q1 = n1 / 8, rem1 = n1 % 8, mine1 = q1 + (die < rem1 ? 1 : 0);
  const int q2 = n2 / 8, rem2 = n2 % 8, mine2 = q2 + (die < rem2 ? 1 : 0);
  if (i >= mine1 + mine2) return;
  int in2;      // how many of the second's tiles stand before this place
  bool second;
  if (first2) {
    in2 = min(i, mine2);
    second = i < mine2;
  } else {
    in2 = (int)((int64_t)i * mine2 / (mine1 + mine2));
    second = (int)((int64_t)(i + 1) * mine2 / (mine1 + mine2)) > in2;
  }
  const int logical = second ? die * q2 + min(die, rem2) + in2 : die * q1 + min(die, rem1) + i - in2;
  if (second) {
    g = g2;
    gx = gx2;
    gy = gy2;
  }
  phases<DUAL, OUT_ACT>(g, logical, gx, gy, rows2, (bf16_t*)smem);
}

static int launch_phases(const MfmaGemmArgs& g, int gy, int64_t n1, const MfmaGemmArgs& g2, int gx2, int gy2, int64_t n2, int rows2, int first2,
                         bool dual, bool out_act, hipStream_t st) {
  const int64_t per_die = (n1 + 7) / 8 + (n2 + 7) / 8;
  if (per_die * 8 > 0x7fffffff) return TQ_ERR_UNSUPPORTED;
  const int shmem = 160 * 1024;      // MI = 2 and 4; 144 KB where MI is 1 or 3
#define TQ_PHASES(D, O)                                                                                                       \
  do {                                                                                                                        \
    if (hipFuncSetAttribute((const void*)gemm_phases_kernel<D, O>, hipFuncAttributeMaxDynamicSharedMemorySize, shmem) != hipSuccess) \
      return TQ_ERR_UNSUPPORTED;                                                                                              \
    hipLaunchKernelGGL((gemm_phases_kernel<D, O>), dim3((unsigned)(per_die * 8)), dim3(512), shmem, st, g, gy, g2, gx2, gy2,  \
                       (int)n2, rows2, first2);                                                                               \
  } while (0)
  if (dual && out_act) TQ_PHASES(true, true);
  else if (dual) TQ_PHASES(true, false);
  else if (out_act) TQ_PHASES(false, true);
  else TQ_PHASES(false, false);
#undef TQ_PHASES
  return 0;
}

// g2 (null: none): a second product, of one matrix and of the same kind, whose tiles fill the chip beside the first's; its k may be
// in runs (k_per, split_stride).
int launch_gemm_phases(const MfmaGemmArgs& g, const MfmaGemmArgs* g2, bool dual, bool out_act, hipStream_t st) {
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
  return launch_phases(g, gy, (int64_t)gx * gy, g2 ? *g2 : g, gx2, gy2, n2, 256, first2, dual, out_act, st);
}

// A product of one matrix, whose rows follow one another, in tiles of `rows` (a multiple of 64 up to 256) rows; k may be in runs.
int launch_gemm_phases_plain(const MfmaGemmArgs& g, int rows, bool dual, bool out_act, hipStream_t st) {
  if (g.tile_group || g.a_rows) return TQ_ERR_BAD_ARG;
  const int cols = dual ? 128 : 256;
  const int64_t gx = (g.M + rows - 1) / rows, gy = (g.N + cols - 1) / cols, n = gx * gy * ((g.K + g.k_per - 1) / g.k_per);
  if (n > (1 << 28)) return TQ_ERR_UNSUPPORTED;
  return launch_phases(g, 1, 0, g, (int)gx, (int)gy, n, rows, 0, dual, out_act, st);
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
