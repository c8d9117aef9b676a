// Matrix products out[m, n] = sum_k a[m, k] * w[n, k] of float operands on the bfloat16 matrix instructions, to the
// accuracy of the float ones.
//
// A float has 24 significant bits, a bfloat16 8 with the same range of exponents: x = h + m + l exactly, h the float
// rounded to bfloat16, m what is left rounded, l the rest.  Of the nine products of two such sums the six of the largest
// terms are added up (h h, h m, m h, m m, h l, l h); those left out (m l, l m, l l) are below 2^-26 of the product, a
// quarter of a float's own rounding.  The sums are float, as in the float instructions.
// Six passes of v_mfma_f32_32x32x16_bf16 cost 6/16 of the float instruction's time: 157 TFLOP/s of float products become
// 400 at the published rates.
#include "gemm_f32.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

#define SPK 32      // k of a step

__device__ __forceinline__ unsigned pack_bf16(float x, float y) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x, y}, bf16x2));
}
__device__ __forceinline__ float low_of(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_of(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

// x = h + m + l, four numbers at a time, two bfloat16 to a word.
__device__ __forceinline__ void split3(const f32x4& x, u32x2& h, u32x2& m, u32x2& l) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float x0 = x[2 * i], x1 = x[2 * i + 1];
    h[i] = pack_bf16(x0, x1);
    const float r0 = x0 - low_of(h[i]), r1 = x1 - high_of(h[i]);
    m[i] = pack_bf16(r0, r1);
    l[i] = pack_bf16(r0 - low_of(m[i]), r1 - high_of(m[i]));
  }
}

// Place of 16-byte chunk q (8 numbers of k) of a row of 64 bytes: eight neighbouring rows' reads of one chunk, and the
// writes of two whole rows, fall on all banks.
__device__ __forceinline__ int split_place(int row, int q) { return row * SPK + ((q ^ ((row >> 1) & 3)) * 8); }

// A tile of 64 MI rows of `a` by 128 rows of w (DUAL: 64 of each matrix) by four waves of 32 MI x 64, 32 of k at a time
// through one LDS buffer of three planes; three workgroups share a compute unit, so that one splits and stages
// while the others multiply.  Bound by the matrix instructions at the clock that they leave: 16,385 x 2,048 times
// 6,144 x 2,048 takes 2.25 ms, 183 TFLOP/s of float products or 1.10 PFLOP/s of bfloat16 ones, where the float
// instructions took 3.42 ms (121 TFLOP/s; the published peak is 157); without the arithmetic of the split 4 % less, so
// that splitting w once ahead would gain little and cost half as much memory again.  Also measured (beside 2.21):
// tiles of 256 rows (two workgroups to a unit) 2.64 ms, steps of k fetched two ahead (two workgroups) 2.32, 16x16x32 instructions 2.83
// (their operands and the next step's rows do not fit the registers of three workgroups).
// The bfloat16 instructions round a sum down, whatever its sign: left alone, every output ends 1.1e-7 of the result's size
// (k 2,048) too low, a shift that all outputs share and that layers behind can carry on.  So every 128 of k the sums and
// the rows of `a` change their sign, and what one block rounds down the next rounds up.
// Against 64 bits the sums are closer than the float instructions': 6.9e-7 of the result against 8.1e-7 at k 2,048, since
// k is rounded into the sum in six steps of 16 where those take eight of 2 (and runs of k make them closer still).
template <int MI, bool DUAL>
__global__ __launch_bounds__(256, MI == 1 ? 4 : 3) void gemm_f32_split_kernel(F32GemmArgs g, int gm, int gn, int k_per_run, float* part) {
  constexpr int BM = 64 * MI, BN = 128, CN = DUAL ? 64 : 128, ROWS = BM + BN, PLANE = ROWS * SPK, FETCH = ROWS / 32;
  __shared__ __align__(16) uint16_t lds[3 * PLANE];
  int m0, n0, group = 0, rows_live;
  if (g.tile_group) {
    // an expert's tiles: items of two units of 64 rows (MI 2) or single units, dealt to the dies in contiguous runs, within
    // an expert column by column
    const int units_all = g.M / 64;
    const int n_units = min(g.n_tiles[0], units_all);
    const int* items = g.tile_group + units_all;
    const int n_items = MI == 2 ? min(g.n_tiles[1], units_all) : n_units;
    const int total = n_items * gn, id = blockIdx.x, die = id % 8, q = total / 8, rem = total % 8;
    if (id / 8 >= q + (die < rem ? 1 : 0)) return;
    const int logical = die * q + min(die, rem) + id / 8;
    const int p = logical / gn;
    auto unit_of = [&](int i) { return MI == 2 ? items[i] : i; };
    group = g.tile_group[unit_of(p)];
    int lo = p, hi = p + 1;
    while (lo > 0 && g.tile_group[unit_of(lo - 1)] == group) --lo;
    while (hi < n_items && g.tile_group[unit_of(hi)] == group) ++hi;
    const int local = logical - lo * gn, item = lo + local % (hi - lo);
    n0 = local / (hi - lo) * CN;
    const int u0 = unit_of(item);
    rows_live = 64 * (MI == 2 && (item + 1 < n_items ? unit_of(item + 1) : n_units) - u0 >= 2 ? 2 : 1);
    m0 = u0 * 64;
  } else {
    // bands of eight row tiles, within a band column by column, a contiguous run of tiles to each die: what a die works on
    // together shares rows of both operands in its L2
    const int total = gm * gn, id = blockIdx.x, die = id % 8, q = total / 8, rem = total % 8;
    const int logical = die * q + min(die, rem) + id / 8;
    const int band = logical / (8 * gn), height = min(8, gm - band * 8), local = logical - band * 8 * gn;
    m0 = (band * 8 + local % height) * BM;
    n0 = local / height * CN;
    rows_live = BM;
  }
  const float* w = g.w + (size_t)group * g.group_stride;
  const float* w2 = DUAL ? g.w2 + (size_t)group * g.group_stride : nullptr;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / 2, wn = wave % 2;
  const int frow = tid / 8, chunk = tid % 8;      // what this thread fetches: rows frow + 32 j, 4 of every 32 of k

  // Rows past the end and rows of padding read some valid row instead: those outputs are never stored.
  const float* src[FETCH];
#pragma unroll
  for (int j = 0; j < FETCH; ++j) {
    const int row = frow + 32 * j;
    if (row < BM) {
      const int m = min(m0 + (row < rows_live ? row : row % 64), g.M - 1);
      src[j] = g.a + (size_t)(g.a_rows && g.a_gather ? max(g.a_rows[m], 0) : m) * g.lda + 4 * chunk;
    } else {
      // (the gated pair: 32 rows of the one matrix, 32 of the other, in turn, so that a wave has both of its columns)
      const int r = row - BM, n = DUAL ? n0 + 32 * (r / 64) + r % 32 : n0 + r;
      src[j] = (DUAL && r / 32 % 2 ? w2 : w) + (size_t)min(n, g.N - 1) * g.K + 4 * chunk;
    }
  }
  const bool active = wm * 32 * MI < rows_live;

  f32x16 acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int k_first = blockIdx.z * k_per_run, k_last = min(g.K, k_first + k_per_run);
  f32x4 next[FETCH];
  unsigned sign = 0;      // of the sums as they stand
  auto negate = [&]() {
    sign ^= 0x80000000u;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = -acc[i][j][v];
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int k0) {
    const bool in = k0 + 4 * chunk < k_last;      // K and the runs are multiples of 4
#pragma unroll
    for (int j = 0; j < FETCH; ++j) next[j] = in ? *reinterpret_cast<const f32x4*>(src[j] + k0) : zero;
  };
  const int r32 = lane % 32, half = lane / 32;
  fetch(k_first);
#pragma unroll 1
  for (int k0 = k_first; k0 < k_last; k0 += SPK) {
    if (k0 > k_first) __syncthreads();
    const unsigned now = ((k0 - k_first) / (4 * SPK) & 1) << 31;
#pragma unroll
    for (int j = 0; j < FETCH; ++j) {
      u32x2 h, m, l;
      if (j < BM / 32)
#pragma unroll
        for (int i = 0; i < 4; ++i) next[j][i] = __uint_as_float(__float_as_uint(next[j][i]) ^ now);
      split3(next[j], h, m, l);
      const int at = split_place(frow + 32 * j, chunk / 2) + 4 * (chunk % 2);
      *reinterpret_cast<u32x2*>(&lds[at]) = h;
      *reinterpret_cast<u32x2*>(&lds[PLANE + at]) = m;
      *reinterpret_cast<u32x2*>(&lds[2 * PLANE + at]) = l;
    }
    __syncthreads();
    if (k0 + SPK < k_last) fetch(k0 + SPK);
    if (active) {
      if (now != sign) negate();
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bf16x8 af[MI][3], wf[2][3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
            af[i][p] = *reinterpret_cast<const bf16x8*>(&lds[p * PLANE + split_place((wm * MI + i) * 32 + r32, 2 * s + half)]);
#pragma unroll
          for (int j = 0; j < 2; ++j)
            wf[j][p] = *reinterpret_cast<const bf16x8*>(&lds[p * PLANE + split_place(BM + (wn * 2 + j) * 32 + r32, 2 * s + half)]);
        }
        // the small terms first; the blocks in turn, so that no instruction waits for the one before it
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PW[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][PA[t]], wf[j][PW[t]], acc[i][j], 0, 0, 0);
      }
    }
  }
  if (!active) return;
  if (sign) negate();

  // Whether this lane has outputs in row v of block i, and those outputs from the two sums behind them (the gated pair's,
  // or of columns 32 apart).
  auto row_of = [&](int i, int v) { return (wm * MI + i) * 32 + 8 * (v / 4) + 4 * half + v % 4; };
  auto live = [&](int i, int v) {
    const int row = row_of(i, v), m = m0 + row;
    return m < g.M && row < rows_live && !(g.a_rows && g.a_rows[m] < 0);
  };
  auto put = [&](int i, int v, float x, float y) {
    const int m = m0 + row_of(i, v), n = n0 + (DUAL ? 32 : 64) * wn + r32;
    if (part) {
      float* to = part + ((size_t)blockIdx.z * g.M + m) * g.N + n;
      if (n < g.N) to[0] = x;
      if (DUAL ? n < g.N : n + 32 < g.N) to[DUAL ? (size_t)gridDim.z * g.M * g.N : 32] = y;
      return;
    }
    float* to = g.out + (size_t)m * g.ldc + n;
    if (DUAL) {
      if (n < g.N) *to = gated_pair(x + f32_bias_at(g, n), y, g.gate, g.limit);
    } else {
      if (n < g.N) to[0] = x + f32_bias_at(g, n);
      if (n + 32 < g.N) to[32] = y + f32_bias_at(g, n + 32);
    }
  };
  unsigned bad[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    bad[i] = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      if (!live(i, v)) continue;
      if (!(fabsf(acc[i][0][v]) <= 3.402823466e38f) || !(fabsf(acc[i][1][v]) <= 3.402823466e38f)) bad[i] |= 1u << v;
      put(i, v, acc[i][0][v], acc[i][1][v]);
    }
  }
  // An operand that is infinite, not a number or beyond the largest bfloat16 has no such split, and leaves a sum that is
  // not finite: those sums are formed again with the float instructions.
#pragma unroll 1
  for (int i = 0; i < MI; ++i) {
    unsigned which = bad[0];
#pragma unroll
    for (int j = 1; j < MI; ++j) which = i == j ? bad[j] : which;
    if (!__any(which != 0)) continue;
    const int row = (wm * MI + i) * 32 + r32, m = min(m0 + (row < rows_live ? row : row % 64), g.M - 1);
    const float* ar = g.a + (size_t)(g.a_rows && g.a_gather ? max(g.a_rows[m], 0) : m) * g.lda;
    const int n = n0 + (DUAL ? 32 : 64) * wn + r32;
    const float* wr = w + (size_t)min(n, g.N - 1) * g.K;
    const float* vr = DUAL ? w2 + (size_t)min(n, g.N - 1) * g.K : w + (size_t)min(n + 32, g.N - 1) * g.K;
    f32x16 x, y;
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] = 0.f, y[v] = 0.f;
#pragma unroll 1
    for (int k = k_first + half; k < k_last; k += 2) {
      x = __builtin_amdgcn_mfma_f32_32x32x2f32(ar[k], wr[k], x, 0, 0, 0);
      y = __builtin_amdgcn_mfma_f32_32x32x2f32(ar[k], vr[k], y, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (which >> v & 1) put(i, v, x[v], y[v]);
  }
}

// Into how many runs of k a product of more than 64 rows is cut: a workgroup's steps of k are a chain of about a
// microsecond each however few workgroups there are, so where the tiles are fewer than two to a compute unit k is cut until
// there are, each run keeping 256 of k at least.  (65 x 2,048 x 2,048: 89 us whole, 30 in four runs; 1,000 x 2,048 x 2,048: 130
// and 67; 2,048 x 2,048 x 5,632, 256 tiles: 363 whole, 276 in two runs, 320 in four; 2,048 x 6,144 x 2,048, 768 tiles: 315 whole,
// 345 in two.)
int f32_split_runs(int M, int N, int K, int* k_per_run) {
  const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
  int64_t runs = 576 / tiles;
  if (runs > K / 256) runs = K / 256;
  if (runs > 8) runs = 8;
  if (runs < 1) runs = 1;
  const int per = (int)((K + runs - 1) / runs + SPK - 1) / SPK * SPK;
  *k_per_run = per;
  return (K + per - 1) / per;
}

int f32_split_product(const F32GemmArgs& g, bool pairs, int runs, int k_per_run, float* part, hipStream_t st) {
  const bool dual = g.w2 != nullptr;
  // tiles of 64 rows where those of 128 would be half empty, or fewer than the compute units
  const int64_t gn = (g.N + (dual ? 63 : 127)) / (dual ? 64 : 128), tall = (int64_t)((g.M + 127) / 128) * gn;
  const bool two = g.tile_group ? pairs : g.M > 128 && tall * runs >= 256;
  const int64_t gm = g.tile_group ? g.M / 64 : two ? (g.M + 127) / 128 : (g.M + 63) / 64;
  if (gm * gn > 0x7fffffff) return TQ_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)(gm * gn), 1, runs), block(256);
#define TQ_SPLIT(MI, D) hipLaunchKernelGGL((gemm_f32_split_kernel<MI, D>), grid, block, 0, st, g, (int)gm, (int)gn, k_per_run, part)
  if (two) {
    if (dual) TQ_SPLIT(2, true);
    else TQ_SPLIT(2, false);
  } else {
    if (dual) TQ_SPLIT(1, true);
    else TQ_SPLIT(1, false);
  }
#undef TQ_SPLIT
  TQ_LAUNCH_CHECK();
  return 0;
}
