// Matrix products out[m, n] = sum_k a[m, k] * w[n, k] in true 32-bit floating point on the matrix cores.
//
// v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32 multiply and add float operands as they are (no reduced-precision
// inputs), at twice the rate that the vector unit reaches without packed instructions.  Same contract as the plain
// product (gemm_generic.hip): optional bias, optional gated pair gate(a w^T) * (a w2^T), optional row gather and
// per-row-tile matrices for experts; the reference's counterpart is its float matvec
// (/root/reference/src/engine/tq_ops.c:296-343).  Two kernels:
//
//  * gemm_f32_tile_kernel, for more than 16 rows: tiles of 64 or 128 rows by 128 columns (64 of most gated pairs) by four
//    waves, 16 of k at a time.  What bounds it is the matrix instructions (64 clocks each), so what counts is that a SIMD always
//    has a wave with products to do: 64 sums a wave and no more, so that three workgroups share a compute unit (two of a
//    gated pair of 64 rows by 128 columns, whose ring is 60 KB, four by 64), and tiles that go
//    straight from memory into a ring of three LDS stages, two on their way, with one bare barrier a tile and no branch around a
//    load (with tiles through registers and loads behind predicates a gated pair of 128 x 128 had one wave to a SIMD).
//    16,385 rows, ms, before and now: by 6,144 x 2,048 3.46 and 3.20 (129 TFLOP/s; the instructions alone give 153), by 2,048 x 5,632 3.48
//    and 3.22, gated pair of twice 5,632 x 2,048 7.55 and 5.78; 60 experts of 1,408 x 2,048, four per token, 6.85 and
//    6.12, their second product 3.80 and 3.22; 1,000 rows by twice 5,632 x 2,048 655 and 402 us.  Rings of two stages 1 to 3 % slower,
//    of four level; four waves to a SIMD (128 registers) level.  Then, with a wave's priority raised while it multiplies (a wave that
//    asks for tiles or has just passed its barrier lets the one in the middle of its products go on), ms without and with: 3.29 and
//    3.15, 3.21 and 3.11, 5.72 and 5.57; experts 6.09 and 6.05, 3.19 and 3.05; 1,000 rows 404 and 388 us.  All of a step's reads
//    before its first product 2 to 4 % slower than a half at a time; waves whose rows all lie behind the last row without their products
//    level to 1 % slower (the loop for each height takes registers that the reads ahead had).
//    17 to 64 rows (a decode step of many sequences) are one row of tiles, at which multiply-adds and bytes of w
//    are in balance; a narrow matrix is cut into runs of k so that the chip has enough workgroups.
//  * gemm_f32_stream_kernel, for few rows (decoding; experts that few tokens chose): the work is reading w once.
//    A workgroup owns 32 rows of w (every row of `a` that a wave fetches multiplies all of them), its four waves split k
//    and add their sums in wave order through LDS; the rows of w go from memory straight into the operand
//    registers, by whole lines of 128 bytes and with the hint that they are read once.
//  Runs of k of a narrow matrix leave their sums apart; a second kernel adds them up in order and finishes them.
//
// A lane's 16 bytes of an operand row are 4 consecutive k, and the four multiply-adds that use them take them one
// by one, so a product sums k in the order (0, 4), (1, 5), (2, 6), (3, 7), (8, 12), ... within each 16 (32x32x2:
// 8 and 16x16x4: 16 elements of k per pass of four instructions); the order depends on k alone, never on the
// row, the number of rows or the tile.
//
// Operand layouts (wave of 64 lanes): 32x32x2: A lane l = row l%32, k l/32; B lane l = column l%32, k l/32; D lane l =
// column l%32, rows 8*(v/4) + 4*(l/32) + v%4, v<16.  16x16x4: A lane l = row l%16, k l/16; B alike; D lane l = column
// l%16, rows 4*(l/16) + v, v<4.
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

// Row of `a` behind output row m, or null.
__device__ __forceinline__ const float* f32_row_of(const F32GemmArgs& g, int m) {
  if (m >= g.M) return nullptr;
  int src = m;
  if (g.a_rows) {
    src = g.a_rows[m];
    if (src < 0) return nullptr;
    if (!g.a_gather) src = m;
  }
  return g.a + (size_t)src * g.lda;
}

// ------------------------------------------------------------------------------------------ many rows
#define TBK 16
#define TSTAGES 3
// Where chunk c (4 of k) of a tile's row lies in the row: eight neighbouring rows' reads of one chunk, and sixteen neighbouring rows'
// where the 64 banks serve them together, fall on banks of their own.
__device__ __forceinline__ int f32_place(int row, int c) { return c ^ (((((row >> 1) ^ (row >> 3)) & 1) << 1) | ((row >> 2) & 1)); }
__device__ __forceinline__ void f32_to_lds16(const float* src, float* wave_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)wave_base, 16, 0, 0);
}

// With `part` set the grid's z cuts k into runs of k_per_split and the sums of run z go to part[z] ([run][M][N], the
// gated pair's second product behind all the first ones) as they are: gemm_f32_reduce_kernel finishes them.
// GO_FIRST: a wave in the middle of its products goes before those of the other workgroups on its SIMD.
template <int MI, int NI, bool DUAL, bool GO_FIRST>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(F32GemmArgs g, int k_per_split, float* part) {
  constexpr int BM = 64 * MI, BN = 64 * NI, ROWS = BM + BN * (DUAL ? 2 : 1), STAGE = ROWS * TBK, L = ROWS / 64;
  __shared__ __align__(16) float ring[TSTAGES * STAGE];
  // Which tile: a die (workgroups are dealt to the 8 of them in turn) gets a contiguous run.  One matrix: bands of 8 row tiles, down
  // a band's columns.  A matrix per expert: expert by expert, within one column by column with its row tiles side by side.
  int tile_m, tile_n;
  {
    const int gx = g.n_tiles ? min(g.n_tiles[0], (int)gridDim.x) : (int)gridDim.x, gy = gridDim.y, total = gx * gy;
    const int id = blockIdx.y * gridDim.x + blockIdx.x, die = id % 8, q = total / 8, rem = total % 8;
    if (id / 8 >= q + (die < rem ? 1 : 0)) return;
    const int logical = die * q + min(die, rem) + id / 8;
    if (g.tile_group) {
      const int at = logical / gy, e = g.tile_group[at], l = threadIdx.x % 64;
      int lo = at, hi = at + 1;
      for (bool more = true; more;) {
        const int c = lo - 1 - l;
        const unsigned long long same = __ballot(c >= 0 && g.tile_group[max(c, 0)] == e);
        lo -= ~same ? __builtin_ctzll(~same) : 64;
        more = !~same;
      }
      for (bool more = true; more;) {
        const int c = hi + l;
        const unsigned long long same = __ballot(c < gx && g.tile_group[min(c, gx - 1)] == e);
        hi += ~same ? __builtin_ctzll(~same) : 64;
        more = !~same;
      }
      const int local = logical - lo * gy;
      tile_n = local / (hi - lo);
      tile_m = lo + local % (hi - lo);
    } else {
      const int band = logical / (8 * gy), in_band = logical % (8 * gy), bh = min(8, gx - band * 8);
      tile_m = band * 8 + in_band % bh;
      tile_n = in_band / bh;
    }
  }
  const int group = g.tile_group ? g.tile_group[tile_m] : 0;
  const float* w = g.w + (size_t)group * g.group_stride;
  const float* w2 = DUAL ? g.w2 + (size_t)group * g.group_stride : nullptr;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wave_m = wave / 2, wave_n = wave % 2;

  // What this thread asks for of each stage: place tid % 4 of rows tid / 4 + 64 i (a's rows, then w's, then w2's).  Rows that do not
  // exist read some valid row instead: those outputs are never stored.
  const float* src[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int r = tid / 4 + 64 * i;      // (a load's 64 rows lie in one of the three: all heights are multiples of 64)
    if (64 * i < BM) {
      const float* from = f32_row_of(g, min(m0 + r, g.M - 1));
      src[i] = from ? from : g.a;
    } else if (64 * i < BM + BN) {
      src[i] = w + (size_t)min(n0 + r - BM, g.N - 1) * g.K;
    } else {
      src[i] = w2 + (size_t)min(n0 + r - BM - BN, g.N - 1) * g.K;
    }
  }
  const int k_first = blockIdx.z * k_per_split, k_last = min(g.K, k_first + k_per_split);
  const int chunk = 4 * f32_place(tid / 4, tid % 4);      // (64 rows on the place is the same)
  auto ask = [&](int step) {
    float* base = ring + step % TSTAGES * STAGE + wave * 16 * TBK;
#pragma unroll
    for (int i = 0; i < L; ++i) f32_to_lds16(src[i] + k_first + step * TBK + chunk, base + 64 * i * TBK);
  };
  // which of this wave's rows exist and are no padding
  const int mw = m0 + wave_m * 32 * MI;
  const unsigned long long live =
      __ballot(lane < 32 * MI && mw + lane < g.M && !(g.a_rows && g.a_rows[min(mw + lane, g.M - 1)] < 0));

  f32x16 acc[MI][NI], acc2[DUAL ? MI : 1][DUAL ? NI : 1];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[i][j][v] = 0.f;
        if (DUAL) acc2[i][j][v] = 0.f;
      }
    }
  const int r32 = lane % 32, kk = lane / 32;
  auto multiply = [&](const float* at) {
    const float* A = at + (wave_m * 32 * MI + r32) * TBK;
    const float* W = at + (BM + wave_n * 32 * NI + r32) * TBK;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = 4 * f32_place(r32, 2 * h + kk);
      f32x4 af[MI], wf[NI], vf[DUAL ? NI : 1];
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = *reinterpret_cast<const f32x4*>(A + i * 32 * TBK + c);
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        wf[j] = *reinterpret_cast<const f32x4*>(W + j * 32 * TBK + c);
        if (DUAL) vf[j] = *reinterpret_cast<const f32x4*>(W + (BN + j * 32) * TBK + c);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][s], wf[j][s], acc[i][j], 0, 0, 0);
            if (DUAL) acc2[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][s], vf[j][s], acc2[i][j], 0, 0, 0);
          }
    }
  };

  const int steps = (k_last - k_first) / TBK, left = (k_last - k_first) % TBK;
  for (int s = 0; s < TSTAGES - 1 && s < steps; ++s) ask(s);
  for (int t = 0; t < steps; ++t) {
    // Tile t has landed once no more of this wave's loads are on their way than those of the tile behind it.  And every wave is
    // through with tile t - 1, whose stage tile t + 2 takes: its reads of it have come back, wherever their products stand.
    if (t + 1 < steps) __builtin_amdgcn_s_waitcnt(0x0070 | L);
    else __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + TSTAGES - 1 < steps) ask(t + TSTAGES - 1);
    if constexpr (GO_FIRST) __builtin_amdgcn_s_setprio(1);
    multiply(ring + t % TSTAGES * STAGE);
    if constexpr (GO_FIRST) __builtin_amdgcn_s_setprio(0);
  }
  if (left) {      // the last 4, 8 or 12 of k, through registers, zeros behind them
    __syncthreads();
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(&ring[(tid / 4 + 64 * i) * TBK + tid % 4 * 4]) =
          chunk < left ? *reinterpret_cast<const f32x4*>(src[i] + k_first + steps * TBK + chunk) : zero;
    }
    __syncthreads();
    multiply(ring);
  }

#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int n = n0 + wave_n * 32 * NI + j * 32 + r32;
    if (n >= g.N) continue;
    const float bias = part ? 0.f : f32_bias_at(g, n);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = i * 32 + 8 * (v / 4) + 4 * kk + v % 4, m = mw + r;
        if (!((live >> r) & 1)) continue;
        if (part) {
          part[((size_t)blockIdx.z * g.M + m) * g.N + n] = acc[i][j][v];
          if (DUAL) part[((size_t)(gridDim.z + blockIdx.z) * g.M + m) * g.N + n] = acc2[i][j][v];
          continue;
        }
        float x = acc[i][j][v] + bias;
        if (DUAL) x = gated_pair(x, acc2[i][j][v], g.gate, g.limit);
        g.out[(size_t)m * g.ldc + n] = x;
      }
  }
}

// ------------------------------------------------------------------------------------------ few rows
__device__ __forceinline__ f32x4 load4_once(const float* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
}
// Lanes l and l ^ 8 (the same quarter q = l / 16, rows r and r ^ 8 of a tile of 16 rows) fetched whole lines of 128
// bytes: lane (r, q) chunk q + 4 (r / 8) of row r % 8 into t0 and of row 8 + r % 8 into t1 (a chunk is 4 floats).
// Afterwards t0 is chunk q and t1 chunk q + 4 of the lane's own row r: the operands of two consecutive passes of 16.
__device__ __forceinline__ void to_own_row(f32x4& t0, f32x4& t1) {
  f32x4 s0, s1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // row_ror:8 reads lane l ^ 8 of each row of 16 lanes; the bank mask says which lanes take it (0xc: 8..15, 0x3: 0..7)
    s0[i] = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(t0[i]), __float_as_int(t1[i]), 0x128, 0xf, 0xc, false));
    s1[i] = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(t1[i]), __float_as_int(t0[i]), 0x128, 0xf, 0x3, false));
  }
  t0 = s0;
  t1 = s1;
}

// A workgroup owns 16 * MT rows of `a` (a row tile of the grid), 16 * NT rows of w (blockIdx.y) and one run of k
// (blockIdx.z, k_per_split long); its four waves take a quarter of the run each.  Every row of `a` that a wave has
// fetched multiplies all 16 * NT rows of w.  With more than one run the sums go to `part` ([run][M][N], the gated
// pair's second product behind all the first ones) as they are, and gemm_f32_reduce_kernel adds the runs up in
// order and finishes them.
template <int MT, int NT, bool DUAL>
__global__ __launch_bounds__(256) void gemm_f32_stream_kernel(F32GemmArgs g, int k_per_split, int k_per_wave, float* part) {
  __shared__ __align__(16) float join[DUAL ? 2 : 1][NT * MT][64 * 4];
  const int tile_m = blockIdx.x, tile_n = blockIdx.y, z = blockIdx.z;
  if (g.n_tiles && tile_m >= g.n_tiles[0]) return;
  const int group = g.tile_group ? g.tile_group[tile_m] : 0;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, q = lane / 16;
  const int m0 = tile_m * 16 * MT, n0 = tile_n * 16 * NT;
  // w is fetched by whole lines: for every 32 of k one instruction takes rows 0..7 of a tile of 16 and the next rows
  // 8..15, eight lanes to a row; lanes r and r ^ 8 then exchange what belongs to the other's row.  A row of w that
  // does not exist reads row 0 instead (what it produces is never stored).
  const int chunk = 4 * (q + 4 * (r / 8));           // this lane's 4 of every 32 of k
  const float* wlo[NT];
  const float* whi[NT];
  const float* vlo[DUAL ? NT : 1];
  const float* vhi[DUAL ? NT : 1];
#pragma unroll
  for (int c = 0; c < NT; ++c) {
    const int n_lo = n0 + 16 * c + r % 8, n_hi = n_lo + 8;
    const size_t o_lo = (size_t)group * g.group_stride + (size_t)(n_lo < g.N ? n_lo : 0) * g.K + chunk;
    const size_t o_hi = (size_t)group * g.group_stride + (size_t)(n_hi < g.N ? n_hi : 0) * g.K + chunk;
    wlo[c] = g.w + o_lo;
    whi[c] = g.w + o_hi;
    if (DUAL) {
      vlo[c] = g.w2 + o_lo;
      vhi[c] = g.w2 + o_hi;
    }
  }
  const float* arow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) arow[t] = f32_row_of(g, m0 + 16 * t + r);

  f32x4 acc[NT][MT], acc2[DUAL ? NT : 1][DUAL ? MT : 1];
#pragma unroll
  for (int c = 0; c < NT; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (DUAL) acc2[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  const int run_end = min(g.K, (z + 1) * k_per_split);
  const int k_beg = z * k_per_split + wave * k_per_wave, k_end = min(run_end, k_beg + k_per_wave);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // P lines of 32 of k whose loads are all issued before the first product
  constexpr int P = (NT * (DUAL ? 2 : 1) * 2 + MT * 2) <= 10 ? 4 : 2;
  for (int k = k_beg; k < k_end; k += 32 * P) {
    f32x4 w0[NT][P], w1[NT][P], v0[DUAL ? NT : 1][DUAL ? P : 1], v1[DUAL ? NT : 1][DUAL ? P : 1], a0[MT][P], a1[MT][P];
    // (a chunk beyond the wave's share is asked for at the matrix's first address instead and replaced by zeros below:
    // every lane loads, so that no load waits behind a branch)
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int kl = k + 32 * p;
      const bool in = kl + chunk < k_end;              // (k_end is a multiple of 4: a chunk lies inside or outside as a whole)
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        w0[c][p] = load4_once(in ? wlo[c] + kl : g.w);
        w1[c][p] = load4_once(in ? whi[c] + kl : g.w);
        if (DUAL) {
          v0[c][p] = load4_once(in ? vlo[c] + kl : g.w2);
          v1[c][p] = load4_once(in ? vhi[c] + kl : g.w2);
        }
      }
      // the rows of `a` stay in cache; they are fetched as the products want them: 4 of k at 4 q of each 16
      const int ka = kl + 4 * q;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        a0[t][p] = *reinterpret_cast<const f32x4*>(ka < k_end && arow[t] ? arow[t] + ka : g.a);
        a1[t][p] = *reinterpret_cast<const f32x4*>(ka + 16 < k_end && arow[t] ? arow[t] + ka + 16 : g.a);
      }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int kl = k + 32 * p;
      const bool in = kl + chunk < k_end;
      const int ka = kl + 4 * q;
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        w0[c][p] = in ? w0[c][p] : zero;
        w1[c][p] = in ? w1[c][p] : zero;
        if (DUAL) {
          v0[c][p] = in ? v0[c][p] : zero;
          v1[c][p] = in ? v1[c][p] : zero;
        }
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        a0[t][p] = ka < k_end && arow[t] ? a0[t][p] : zero;
        a1[t][p] = ka + 16 < k_end && arow[t] ? a1[t][p] : zero;
      }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        to_own_row(w0[c][p], w1[c][p]);
        if (DUAL) to_own_row(v0[c][p], v1[c][p]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < NT; ++c)
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0[c][p][i], a0[t][p][i], acc[c][t], 0, 0, 0);
            if (DUAL) acc2[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0[c][p][i], a0[t][p][i], acc2[c][t], 0, 0, 0);
          }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < NT; ++c)
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[c][p][i], a1[t][p][i], acc[c][t], 0, 0, 0);
            if (DUAL) acc2[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1[c][p][i], a1[t][p][i], acc2[c][t], 0, 0, 0);
          }
    }
  }
  // the waves' sums are added in wave order: waves 1, 2, 3 hand theirs to wave 0 one after the other
  for (int ww = 1; ww < 4; ++ww) {
    if (wave == ww) {
#pragma unroll
      for (int c = 0; c < NT; ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          *reinterpret_cast<f32x4*>(&join[0][c * MT + t][lane * 4]) = acc[c][t];
          if (DUAL) *reinterpret_cast<f32x4*>(&join[DUAL ? 1 : 0][c * MT + t][lane * 4]) = acc2[c][t];
        }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int c = 0; c < NT; ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          acc[c][t] += *reinterpret_cast<const f32x4*>(&join[0][c * MT + t][lane * 4]);
          if (DUAL) acc2[c][t] += *reinterpret_cast<const f32x4*>(&join[DUAL ? 1 : 0][c * MT + t][lane * 4]);
        }
    }
    __syncthreads();
  }
  if (wave != 0) return;
  const bool raw = part != nullptr;       // several runs of k: leave the sums as they are
  float* dst = raw ? part + (size_t)z * g.M * g.N : g.out;
  const int64_t ld = raw ? g.N : g.ldc;
#pragma unroll
  for (int c = 0; c < NT; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      // D: lane = column (row of `a`) r, rows (rows of w) 4 q + v
      const int m = m0 + 16 * t + r;
      if (m >= g.M) continue;
      if (g.a_rows && g.a_rows[m] < 0) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int nn = n0 + 16 * c + 4 * q + v;
        if (nn >= g.N) continue;
        if (raw) {
          dst[(size_t)m * ld + nn] = acc[c][t][v];
          if (DUAL) dst[(size_t)gridDim.z * g.M * g.N + (size_t)m * ld + nn] = acc2[c][t][v];
        } else {
          float x = acc[c][t][v] + f32_bias_at(g, nn);
          if (DUAL) x = gated_pair(x, acc2[c][t][v], g.gate, g.limit);
          dst[(size_t)m * ld + nn] = x;
        }
      }
    }
}

// out[m][n] = sum over the runs, in order, of part[run][m][n] (+ bias; the gated pair: gate(that) * the same sum of
// the second product's runs).  With `keep_runs` the runs stay apart and only the bias is added, to run 0.
__global__ void gemm_f32_reduce_kernel(F32GemmArgs g, const float* __restrict__ part, int S, int dual) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)g.M * g.N) return;
  const int m = (int)(i / g.N), n = (int)(i % g.N);
  float x = 0.f, y = 0.f;
  for (int z = 0; z < S; ++z) {
    x += part[(size_t)z * g.M * g.N + i];
    if (dual) y += part[(size_t)(S + z) * g.M * g.N + i];
  }
  x += f32_bias_at(g, n);
  if (dual) x = gated_pair(x, y, g.gate, g.limit);
  g.out[(size_t)m * g.ldc + n] = x;
}
__global__ void gemm_f32_bias_kernel(F32GemmArgs g) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)g.M * g.N) return;
  g.out[i] += f32_bias_at(g, (int)(i % g.N));
}

// Into how many runs k is cut for a plain product (one matrix, up to 64 rows): enough that a narrow matrix still
// gives every compute unit two workgroups (of 128 columns for 17 to 64 rows, of 32 for fewer), each run keeping at
// least 256 of k.  A function of N and K alone, so that a row's sums do not depend on how many rows there are.
// Tiles of 16 rows of w per workgroup of the few-row kernel.  Measured on the experts' gated product at 64, 128 and 240
// tokens (60 experts of 1,408 x 2,048, 4 per token): 290, 299 and 412 us with 2; 315, 317 and 436 with 4; 272, 289 and 423 with 1.
#define SNT 2
static int f32_runs_of_k(int N, int K, int* k_per_split) {
  const int groups = (N + 127) / 128;
  int runs = 1;
  while (runs < 32 && groups * runs < 512 && K / (runs * 2 * 4 * 16) >= 2) runs *= 2;
  int per = ((K + runs - 1) / runs + 127) / 128 * 128;    // a multiple of 128: a quarter for each wave, in whole lines
  if (per < 128) per = 128;
  *k_per_split = per;
  return (K + per - 1) / per;
}
TQ_API int tq_gemm_f32_runs(int M, int N, int K, int grouped) {
  int per;
  return (grouped || M > 64) ? 1 : f32_runs_of_k(N, K, &per);      // (grouped: also a product whose rows are gathered)
}

// tile_rows: 16 or 64 rows of output per row tile; with tile_group set it is the padding unit that the row order
// was built with.  K must be a multiple of 4 and every row of a, w and w2 must start at a multiple of 16 bytes.
// scratch: for a plain product of up to 64 rows, tq_gemm_f32_runs(M, N, K, 0) * M * N floats (twice that for a gated
// pair), unless that number is 1.  keep_runs (plain products into which no second matrix goes): `out` is
// [runs][M][N] and receives the runs apart, the bias in run 0; the caller adds them up in order.
TQ_API int tq_gemm_f32(const void* a, int64_t lda, const int* a_rows, int a_gather, const void* w, const void* w2,
                       int64_t group_stride, const int* tile_group, const int* n_tiles, const void* bias, int bias_type,
                       void* out, int64_t ldc, int M, int N, int K, int tile_rows, int gate, void* scratch, int keep_runs,
                       hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (tile_rows != 16 && tile_rows != 64)) return TQ_ERR_BAD_ARG;
  if (K % 4 != 0 || lda % 4 != 0 || group_stride % 4 != 0 || ((size_t)a & 15) || ((size_t)w & 15) || ((size_t)w2 & 15))
    return TQ_ERR_UNSUPPORTED;
  if (gate < 0 || gate >= TQ_GATE_COUNT) return TQ_ERR_BAD_ARG;
  F32GemmArgs g{(const float*)a, lda, a_rows, a_gather, (const float*)w, (const float*)w2, group_stride, tile_group,
                n_tiles, bias, bias_type, (float*)out, ldc, M, N, K, gate, tq_pair_limit_host};
  const bool dual = w2 != nullptr;
  const bool grouped = tile_group != nullptr;
  if (keep_runs && (dual || grouped || a_rows || ldc != N)) return TQ_ERR_BAD_ARG;
  int k_per_split = (K + 127) / 128 * 128;
  const int runs = (grouped || a_rows || M > 64) ? 1 : f32_runs_of_k(N, K, &k_per_split);
  float* part = nullptr;
  if (runs > 1) {
    part = keep_runs ? (float*)out : (float*)scratch;
    if (!part) return TQ_ERR_BAD_ARG;
  }
  if ((grouped && tile_rows == 16) || (!grouped && M <= 16)) {
    // few rows: the work is reading w once
    const int k_per_wave = k_per_split / 4;
    const dim3 grid((M + 15) / 16, (N + 16 * SNT - 1) / (16 * SNT), runs);
    if (grid.y > 65535) return TQ_ERR_UNSUPPORTED;
    if (dual)
      hipLaunchKernelGGL((gemm_f32_stream_kernel<1, SNT, true>), grid, dim3(256), 0, st, g, k_per_split, k_per_wave, part);
    else
      hipLaunchKernelGGL((gemm_f32_stream_kernel<1, SNT, false>), grid, dim3(256), 0, st, g, k_per_split, k_per_wave, part);
  } else {
    // tiles; 17 to 64 rows of one matrix are a single row of tiles, cut into runs of k where the matrix is narrow.  A gated pair of
    // more rows goes in tiles of 128 rows by 64 columns, as long as the grid's y has room for as many (4,194,240 columns of either
    // matrix), beyond that in tiles of 64 rows, whose sums run over k alike.
    // A gated pair in tiles of 64 rows: by 128 columns two workgroups share a compute unit, by 64 columns four, but `a` passes twice as
    // often.  64 columns while the tiles of 128 are within five rounds of those two (us by 128 and by 64 columns: 24 rows by twice 6,144
    // x 2,048 58 and 48, 64 by 20,480 x 3,584 250 and 203; 60 experts of 1,408 x 2,048, four per token, 250 tokens 523 and 429, 2,000
    // (2,035 tiles) 1,035 and 979, 3,000 (2,717) 1,338 and 1,381, 18,000 6,550 and 6,901; 32 of 4,096 x 2,048, two per token, 2,000
    // tokens (3,008) 1,359 and 1,406; 8 of 4,096 x 1,024 3,000 tokens (3,264) 898 and 863).
    const bool fits = (N + 63) / 64 <= 65535;
    const int mi = (grouped || M <= 64 || (dual && !fits)) ? 1 : 2;
    const bool narrow = dual && fits && (mi == 2 || (int64_t)((M + 63) / 64) * ((N + 127) / 128) <= 5 * 512);
    const int columns = narrow ? 64 : 128;
    const dim3 grid((M + 64 * mi - 1) / (64 * mi), (N + columns - 1) / columns, runs);
    if (grid.y > 65535) return TQ_ERR_UNSUPPORTED;
    // A wave's priority where workgroups share SIMDs, that is more than one to a compute unit, and not where one row of tiles waits for w.
    // Three to a unit are a round of 768; up to three rounds whose last leaves more than a quarter of the chip empty go without, since those
    // that go first leave the others of their unit behind, which then end alone (times with it over without, 17 to 4,096 rows by 2,048 to
    // 32,000 columns, k 512 to 5,632: up to 256 workgroups 1.01 to 1.03, to 768 0.96 to 1.00; 1,000 to 1,024 1.00 to 1.14, 2,000 to 2,048 1.04 to
    // 1.10; 1,376 and 1,536 0.96 to 0.98, 2,752 and more 0.97 to 1.00 (two of 30 1.02 and 1.06); one row of tiles of a gated pair up to 1.08).
    const int64_t n = (int64_t)grid.x * grid.y;      // (of experts: at most)
    const bool first = grid.x > 1 && n > 256 && (grouped || n <= 768 || n >= 3 * 768 || n % 768 == 0 || n % 768 >= 576);
#define TQ_F32_TILE(...)                                                                                                     \
  do {                                                                                                                       \
    if (first) hipLaunchKernelGGL((gemm_f32_tile_kernel<__VA_ARGS__, true>), grid, dim3(256), 0, st, g, k_per_split, part);  \
    else hipLaunchKernelGGL((gemm_f32_tile_kernel<__VA_ARGS__, false>), grid, dim3(256), 0, st, g, k_per_split, part);       \
  } while (0)
    if (mi == 1) {
      if (narrow) TQ_F32_TILE(1, 1, true);
      else if (dual) TQ_F32_TILE(1, 2, true);
      else TQ_F32_TILE(1, 2, false);
    } else {
      if (dual) TQ_F32_TILE(2, 1, true);
      else TQ_F32_TILE(2, 2, false);
    }
#undef TQ_F32_TILE
  }
  if (runs > 1) {
    const unsigned blocks = (unsigned)(((int64_t)M * N + 255) / 256);
    if (!keep_runs)
      hipLaunchKernelGGL(gemm_f32_reduce_kernel, dim3(blocks), dim3(256), 0, st, g, part, runs, dual ? 1 : 0);
    else if (bias)
      hipLaunchKernelGGL(gemm_f32_bias_kernel, dim3(blocks), dim3(256), 0, st, g);
  }
  TQ_LAUNCH_CHECK();
  return 0;
}
