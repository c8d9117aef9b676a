// Matrix products out[m, n] = sum_k a[m, k] * w[n, k] on the matrix cores, bfloat16 in, float sums.
//
// Same contract as the plain product (gemm_generic.hip): optional bias, optional gated pair gate(a w^T) * (a w2^T)
// (gate: silu or another activation), optional row gather and per-row-tile matrices for experts.  The kernels:
//
//  * gemm_stream_kernel, for few rows (decoding): the work is reading w once.  A wave owns 16 rows of w
//    and streams them straight from memory into the operand registers of v_mfma_f32_16x16x32_bf16 (lane
//    l holds 8 consecutive k of row l % 16).  The loads take whole lines of 128 bytes, eight lanes to a row, with
//    the hint that the bytes are read once, and pairs of lanes then exchange registers: half lines per
//    instruction, which the operand layout would give by itself, read a quarter slower.  The few rows of `a`
//    are read the same way, without the hint, and stay in cache.  The waves of a workgroup split k among them and
//    add their partial sums in wave order through LDS, so that even a narrow matrix gives the chip enough
//    waves and bytes in flight.  How k is split depends on N and K only, never on the number of rows.
//    gemm_lean_kernel is the same for whole lines of k and whole tiles of columns, which nearly all products are.
//  * gemm_tile_kernel, for many rows (prompts): tiles of BM x 128 outputs by eight waves, 64 of k at a time staged
//    through two LDS buffers (16-byte chunks, XOR-swizzled by row so that the operand reads of
//    v_mfma_f32_32x32x16_bf16 do not collide); while one buffer is multiplied the next tile is written into
//    the other and the one after that is on its way from memory.
//  * gemm_few_tiles_kernel, for up to some hundred rows of one matrix: smaller tiles through a ring of LDS buffers, the same sums.
//  * gemm_phases_kernel (gemm_phases.hip), for experts with many rows and for many rows of one matrix where k is in whole tiles: tiles
//    of up to 256 x 256, the same sums.
//
// Operand layouts (wave of 64 lanes): 16x16x32: A lane l = row l%16, k 8*(l/16)..+7; B lane l = column l%16,
// same k; D lane l = column l%16, rows 4*(l/16)+v, v<4.  32x32x16: A lane l = row l%32, k 8*(l/32)..+7;
// B alike; D lane l = column l%32, rows 8*(v/4) + 4*(l/32) + v%4, v<16.
#include "common.h"

#include "gemm_mfma.h"
#include <string.h>

// ------------------------------------------------------------------------------------------ few rows
// The sums of one wave: its share k_beg .. k_end of k for NTL tiles of 16 columns (tile t starts at column col0[t])
// and MT tiles of 16 rows (ap: the rows of `a` that this lane fetches, q: its chunk of 8 within each 64 of k).
template <int MT, bool DUAL, int NTL>
__device__ __forceinline__ void stream_accumulate(const MfmaGemmArgs& g, const int (&col0)[NTL], int group,
                                                  const bf16_t* const (&ap)[MT][2], int q, int k_beg, int k_end,
                                                  f32x4 (&acc)[NTL][MT], f32x4 (&acc2)[DUAL ? NTL : 1][DUAL ? MT : 1]) {
  const int r = (threadIdx.x % 64) % 16;
#pragma unroll
  for (int t = 0; t < NTL; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (DUAL) acc2[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  // U steps of 32 at a time, every load issued before the first product, so that a wave keeps U (2U with the
  // gated pair) kilobytes of w in flight per column tile.  w and a are fetched by whole lines: for each pair of
  // steps (64 of k, 128 bytes of a row) eight lanes take a row, one instruction the tile's rows 0..7 and the next
  // rows 8..15, and lanes l and l ^ 8 then exchange what belongs to the other's row.  Rows of w that do not exist
  // read row 0 instead (what they produce is never stored); rows of a that do not exist, and chunks beyond the
  // wave's share or beyond K, load nothing and multiply zeros.
  constexpr int U_ONE = (DUAL ? 4 : 8) / (MT == 4 ? 2 : 1);
  constexpr int U = U_ONE / NTL >= 2 ? U_ONE / NTL : 2;
  {
    size_t row_a[NTL], row_b[NTL];
#pragma unroll
    for (int t = 0; t < NTL; ++t) {
      const int n_a = col0[t] + r % 8, n_b = n_a + 8;
      row_a[t] = (size_t)group * g.group_stride + (size_t)(n_a < g.N ? n_a : 0) * g.K + q * 8;
      row_b[t] = (size_t)group * g.group_stride + (size_t)(n_b < g.N ? n_b : 0) * g.K + q * 8;
    }
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int k = k_beg; k < k_end; k += 32 * U) {
      u32x4 wf[NTL][U], vf[DUAL ? NTL : 1][DUAL ? U : 1];
      u32x4 af[MT][U];
#pragma unroll
      for (int j = 0; j < U / 2; ++j) {
        const int kp = k + 64 * j;
        const bool okw = kp + q * 8 < k_end;      // k_end <= K, both multiples of 8: a chunk is in or out as a whole
#pragma unroll
        for (int t = 0; t < NTL; ++t) {
          wf[t][2 * j] = okw ? load16_once(g.w + row_a[t] + kp) : zero;
          wf[t][2 * j + 1] = okw ? load16_once(g.w + row_b[t] + kp) : zero;
          if (DUAL) {
            vf[t][2 * j] = okw ? load16_once(g.w2 + row_a[t] + kp) : zero;
            vf[t][2 * j + 1] = okw ? load16_once(g.w2 + row_b[t] + kp) : zero;
          }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int hf = 0; hf < 2; ++hf)
            af[mt][2 * j + hf] = okw && ap[mt][hf] ? *reinterpret_cast<const u32x4*>(ap[mt][hf] + kp) : zero;
      }
#pragma unroll
      for (int j = 0; j < U / 2; ++j) {
#pragma unroll
        for (int t = 0; t < NTL; ++t) {
          to_own_row(wf[t][2 * j], wf[t][2 * j + 1]);
          if (DUAL) to_own_row(vf[t][2 * j], vf[t][2 * j + 1]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) to_own_row(af[mt][2 * j], af[mt][2 * j + 1]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const bf16x8 ax = __builtin_bit_cast(bf16x8, af[mt][u]);
#pragma unroll
          for (int t = 0; t < NTL; ++t) {
            acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax, __builtin_bit_cast(bf16x8, wf[t][u]), acc[t][mt], 0, 0, 0);
            if (DUAL)
              acc2[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax, __builtin_bit_cast(bf16x8, vf[t][u]), acc2[t][mt], 0, 0, 0);
          }
        }
    }
  }
}

// A workgroup of 64 * (waves that split k) threads takes column tile `tile_n` (16 * NTL columns) of row tile
// `tile_m` (16 * MT rows) over run `z` of k (k_per long; run 0 is all of k unless the product is split into
// partial sums); red: LDS of [waves][NTL * MT * (DUAL ? 2 : 1)][4][64] floats.  What a wave reads of `a` serves
// its NTL tiles of 16 columns: with many rows the way of `a` from L2 into the compute unit is what binds, and two
// column tiles per wave halve it.
template <int MT, bool DUAL, bool OUT_ACT, int NTL = 1>
__device__ __forceinline__ void stream_body(MfmaGemmArgs g, int tile_n, int tile_m, int z, float* red) {
  if (g.n_tiles && tile_m >= g.n_tiles[0]) return;
  const int k_lo = z * g.k_per, k_hi = min(g.K, k_lo + g.k_per);
  if (z) {
    g.out = (float*)g.out + z * g.split_stride;
    g.bias = nullptr;
  }
  const int group = g.tile_group ? g.tile_group[tile_m] : 0;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, nw = blockDim.x / 64;
  const int r = lane % 16, c = lane / 16;
  const int n0 = tile_n * 16 * NTL, m0 = tile_m * 16 * MT;
  // the rows of `a` that this lane fetches: r % 8 and 8 + r % 8 of each tile of 16 (as with w below)
  const int q = c + 4 * (r / 8);            // and the chunk of 8 within each 64 of k
  const bf16_t* ap[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int m = m0 + mt * 16 + 8 * hf + r % 8;
      int src = -1;
      if (m < g.M) {
        src = g.a_rows ? g.a_rows[m] : m;
        if (src >= 0 && !g.a_gather) src = m;
      }
      ap[mt][hf] = src >= 0 ? g.a + (size_t)src * g.lda + q * 8 : nullptr;
    }
  // this wave's share of k, in steps of 32; an even number of them, so that every pair of steps is a line of w
  const int steps = (k_hi - k_lo + 31) / 32;
  const int per = ((steps + nw - 1) / nw + 1) & ~1;
  const int k_beg = k_lo + wave * per * 32, k_end = min(k_hi, k_lo + (wave + 1) * per * 32);

  f32x4 acc[NTL][MT], acc2[DUAL ? NTL : 1][DUAL ? MT : 1];
  int col0[NTL];
#pragma unroll
  for (int t = 0; t < NTL; ++t) col0[t] = n0 + 16 * t;
  stream_accumulate<MT, DUAL, NTL>(g, col0, group, ap, q, k_beg, k_end, acc, acc2);
  // The waves' partial sums are added in wave order, every thread of the workgroup taking some of the outputs.
  constexpr int PAIRS = NTL * MT;               // (column tile, row tile) pairs: set t * MT + mt, the gate's partner PAIRS on
  constexpr int SETS = PAIRS * (DUAL ? 2 : 1);
  if (nw > 1) {
#pragma unroll
    for (int t = 0; t < NTL; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          red[((wave * SETS + t * MT + mt) * 4 + v) * 64 + lane] = acc[t][mt][v];
          if (DUAL) red[((wave * SETS + PAIRS + t * MT + mt) * 4 + v) * 64 + lane] = acc2[t][mt][v];
        }
    __syncthreads();
    for (int i = threadIdx.x; i < PAIRS * 256; i += blockDim.x) {
      const int ol = i % 64, v = (i / 64) % 4, pair = i / 256, mt = pair % MT, t = pair / MT;
      float s = 0.f, s2 = 0.f;
      for (int w = 0; w < nw; ++w) {
        s += red[((w * SETS + pair) * 4 + v) * 64 + ol];
        if (DUAL) s2 += red[((w * SETS + PAIRS + pair) * 4 + v) * 64 + ol];
      }
      const int on = n0 + 16 * t + ol % 16, om = m0 + mt * 16 + 4 * (ol / 16) + v;
      if (on >= g.N || om >= g.M) continue;
      if (g.a_rows && g.a_rows[om] < 0) continue;
      float o = s + bias_at(g, on);
      if (DUAL) o = gated_pair(o, s2, g.gate, g.limit);
      store_out<OUT_ACT>(g, om, on, o);
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < NTL; ++t) {
    const int n = n0 + 16 * t + r;
    if (n >= g.N) continue;
    const float b = bias_at(g, n);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = m0 + mt * 16 + 4 * c + v;
        if (m >= g.M) continue;
        if (g.a_rows && g.a_rows[m] < 0) continue;
        float o = acc[t][mt][v] + b;
        if (DUAL) o = gated_pair(o, acc2[t][mt][v], g.gate, g.limit);
        store_out<OUT_ACT>(g, m, n, o);
      }
  }
}

// grid (ceil(N / (16 NTL)), row tiles of 16 * MT rows, runs of k).  Two column tiles per wave need the registers of a
// workgroup of at most 8 waves.
template <int MT, bool DUAL, bool OUT_ACT, int NTL>
__global__ __launch_bounds__(NTL > 1 ? 512 : 1024) void gemm_stream_kernel(MfmaGemmArgs g) {
  extern __shared__ float red[];
  stream_body<MT, DUAL, OUT_ACT, NTL>(g, blockIdx.x, blockIdx.y, blockIdx.z, red);
}

// Two products that do not depend on each other in one launch (decoding: the routed experts' product beside
// the shared expert's): workgroups 0 .. n2 - 1 take the second, smaller one (column tile id % nx2 of row tile
// id / nx2 % rows2, run id / nx2 / rows2 of k), so that it is under way at once, the others the first.  Both are
// split over k by the waves of this launch; the second one, when its k is much longer than the first one's, also
// into runs whose partial sums go out apart.
template <bool DUAL, bool OUT_ACT>
__global__ __launch_bounds__(1024) void gemm_stream_pair_kernel(MfmaGemmArgs g1, int nx1, MfmaGemmArgs g2, int nx2,
                                                                 int rows2, int n2) {
  extern __shared__ float red[];
  const int id = blockIdx.x;
  if (id < n2)
    stream_body<1, DUAL, OUT_ACT>(g2, id % nx2, id / nx2 % rows2, id / nx2 / rows2, red);
  else
    stream_body<1, DUAL, OUT_ACT>(g1, (id - n2) % nx1, (id - n2) / nx1, 0, red);
}

// ------------------------------------------------------------------------------------------ few rows, whole lines
// The streaming kernel for what nearly every product of a decode step is: k in whole lines of 64, columns in whole tiles of 16, up to
// 16 rows a tile.  Same sums in the same order as stream_body, so the same bits, but no lane asks whether its chunk or its row is
// there: a row that is none reads the tile's first row instead (what it gives is never stored: a row of the product depends on its
// own row of `a` alone), and a last round with fewer lines is a branch of the whole wave.
//
// What bounds it: the matrices' way from memory, and for the small ones what a launch and a wave's chain of first load, products, LDS
// and store take.  Every load a branch of its own, as stream_body has them, kept the last of a round from being asked for until the
// first had come, and cost a microsecond of 5 to 9.
// Measured, us a launch in a captured graph, one row: 2,048 x 2,048 5.4 -> 4.4 (a plain read of its bytes: 3.6), 2,048 x 5,632 9.1 ->
// 6.8, a gated pair of 5,632 x 2,048 12.6 -> 10.4 (read: 8.8), four of 60 experts' pairs of 1,408 x 2,048 12.3 -> 10.6 and second
// products 8.3 -> 6.7, 32,000 x 2,048 24.2 -> 22.5.  Asking for more lines at once (R) made large products slower: 4 KB of every stream
// and wave fill the path.
//
// NT streams of COLS columns (1, or a gated pair's two matrices), wb[t] their first line of this wave's share, `lines` lines of 64 of
// k.  A lane's loads are whole lines as above.  COLS 8: the operands of columns 8..15 are other columns' and nothing is stored of
// them.  A8: the tile has no row behind its eighth, so `a` is read as such a w is (ap: row r % 8, chunk q); else in the operands' own
// layout (ap: row r, chunk c).
// v of lane l ^ 8
__device__ __forceinline__ u32x4 from_other_half(const u32x4& v) {
  u32x4 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = __builtin_amdgcn_update_dpp(0, v[i], 0x128, 0xf, 0xf, false);      // row_ror:8
  return s;
}
// row of lane l % 8 of its 16
__device__ __forceinline__ int row_of_eight(int row) { return __builtin_amdgcn_update_dpp(row, row, 0x128, 0xf, 0xc, false); }
typedef const __attribute__((address_space(1))) char* global_bytes;
typedef const __attribute__((address_space(1))) u32x4* global_u32x4;
template <int COLS, int NT, int R, bool A8, bool FULL>
__device__ __forceinline__ void lean_round(const global_bytes (&wb)[NT], unsigned off, unsigned off8, global_bytes ap, int lines,
                                           f32x4 (&acc)[NT]) {
  u32x4 wf[NT][R][COLS / 8], af[R][2];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (!FULL && j && j >= lines) break;
    af[j][0] = *(global_u32x4)(ap + 128 * j);
    if (!A8) af[j][1] = *(global_u32x4)(ap + 128 * j + 64);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      wf[t][j][0] = __builtin_nontemporal_load((global_u32x4)(wb[t] + off + 128 * j));
      if (COLS > 8) wf[t][j][COLS / 8 - 1] = __builtin_nontemporal_load((global_u32x4)(wb[t] + off8 + 128 * j));
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (!FULL && j && j >= lines) break;
    if (A8) af[j][1] = from_other_half(af[j][0]);
    u32x4 second[NT];      // the operand of the line's second half
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (COLS > 8) {
        to_own_row(wf[t][j][0], wf[t][j][COLS / 8 - 1]);
        second[t] = wf[t][j][COLS / 8 - 1];
      } else {
        second[t] = from_other_half(wf[t][j][0]);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[j][h]),
                                                         __builtin_bit_cast(bf16x8, h ? second[t] : wf[t][j][0]), acc[t], 0, 0, 0);
  }
}
template <int COLS, int NT, int R, bool A8>
__device__ __forceinline__ void lean_accumulate(global_bytes (&wb)[NT], unsigned off, unsigned off8, global_bytes ap, int lines,
                                                f32x4 (&acc)[NT]) {
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (; lines >= R; lines -= R) {
    lean_round<COLS, NT, R, A8, true>(wb, off, off8, ap, R, acc);
#pragma unroll
    for (int t = 0; t < NT; ++t) wb[t] += 128 * R;
    ap += 128 * R;
  }
  if (lines > 0) lean_round<COLS, NT, R, A8, false>(wb, off, off8, ap, lines, acc);
}

// One workgroup's COLS columns of tile `tile_m` (run z of k); GROUP: a matrix per row tile, by the row order's lists.
template <bool DUAL, bool OUT_ACT, bool GROUP, int COLS>
__device__ __forceinline__ void lean_body(const MfmaGemmArgs& g, int tile_n, int tile_m, int z, float* red) {
  constexpr int NT = DUAL ? 2 : 1, R = 4 / NT;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), nw = blockDim.x / 64;
  const int r = lane % 16, c = lane / 16, q = c + 4 * (r / 8);
  const int m0 = GROUP ? tile_m * 16 : 0, n0 = tile_n * COLS;
  // which matrix and which rows, asked for together
  const int live_tiles = GROUP ? g.n_tiles[0] : 1, group = GROUP ? g.tile_group[tile_m] : 0;
  const int src = GROUP ? g.a_rows[m0 + r] : r < g.M ? r : -1;
  if (GROUP) asm volatile("" ::"s"(group), "v"(src));
  if (GROUP && tile_m >= live_tiles) return;
  const unsigned live = (unsigned)__ballot(src >= 0) & 0xffff;
  const int own = !GROUP || g.a_gather ? src : m0 + r;
  const int first = __builtin_amdgcn_readfirstlane(own);      // (by all lanes: lane 0 has the tile's first row, which is never padding)
  const int row = max(src >= 0 ? own : first, 0);
  const int k_lo = z * g.k_per, k_hi = min(g.K, k_lo + g.k_per);
  const int steps = (k_hi - k_lo + 31) / 32, per = ((steps + nw - 1) / nw + 1) & ~1;
  const int k_beg = k_lo + wave * per * 32, lines = (min(k_hi, k_beg + per * 32) - k_beg) / 64;
  global_bytes wb[NT];
  wb[0] = (global_bytes)(g.w + (size_t)group * g.group_stride + (size_t)n0 * g.K + k_beg);
  if (DUAL) wb[NT - 1] = (global_bytes)(g.w2 + (size_t)group * g.group_stride + (size_t)n0 * g.K + k_beg);
  const unsigned off = ((unsigned)(r % 8) * g.K + q * 8) * 2;
  f32x4 acc[NT];
  if (live >> 8)
    lean_accumulate<COLS, NT, R, false>(wb, off, off + 16 * g.K, (global_bytes)(g.a + (size_t)row * g.lda + k_beg + 8 * c), lines, acc);
  else
    lean_accumulate<COLS, NT, R, true>(wb, off, off + 16 * g.K, (global_bytes)(g.a + (size_t)row_of_eight(row) * g.lda + k_beg + 8 * q), lines, acc);
  float* out = (float*)g.out + z * g.split_stride;      // (runs of k go out as floats)
  auto store = [&](int i, float s, float s2) {
    const int on = n0 + i % 16, om = 4 * (i % 64 / 16) + i / 64;
    if ((COLS < 16 && i % 16 >= COLS) || !((live >> om) & 1)) return;
    float o = s + (z ? 0.f : bias_at(g, on));
    if (DUAL) o = gated_pair(o, s2, g.gate, g.limit);
    if (g.act1) o = gate_fn(o, g.act1 - 1);
    const size_t at = (size_t)(m0 + om) * g.ldc + on;
    if (OUT_ACT) ((bf16_t*)g.out)[at] = f32_to_bf16(o);
    else out[at] = o;
  };
  if (nw > 1) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((wave * NT + t) * 4 + v) * 64 + lane] = acc[t][v];
    __syncthreads();
    for (int i = threadIdx.x; i < 256; i += blockDim.x) {
      float s = 0.f, s2 = 0.f;
      for (int w = 0; w < nw; w += 2) {      // (an even number of waves)
        const float* at = red + w * NT * 256 + i;
        const float a0 = at[0], a1 = at[NT * 256], b0 = DUAL ? at[256] : 0.f, b1 = DUAL ? at[NT * 256 + 256] : 0.f;
        s += a0;
        s += a1;
        if (DUAL) {
          s2 += b0;
          s2 += b1;
        }
      }
      store(i, s, s2);
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) store(v * 64 + lane, acc[0][v], acc[NT - 1][v]);
  }
}

template <bool DUAL, bool OUT_ACT, bool GROUP, int COLS>
__global__ __launch_bounds__(1024) void gemm_lean_kernel(MfmaGemmArgs g) {
  extern __shared__ float red[];
  lean_body<DUAL, OUT_ACT, GROUP, COLS>(g, blockIdx.x, blockIdx.y, blockIdx.z, red);
}
// (as gemm_stream_pair_kernel; the first over experts, the second of one matrix)
template <bool DUAL, bool OUT_ACT, int COLS>
__global__ __launch_bounds__(1024) void gemm_lean_pair_kernel(MfmaGemmArgs g1, int nx1, MfmaGemmArgs g2, int nx2, int n2) {
  extern __shared__ float red[];
  const int id = blockIdx.x;
  if (id < n2) lean_body<DUAL, OUT_ACT, false, COLS>(g2, id % nx2, 0, id / nx2, red);
  else lean_body<DUAL, OUT_ACT, true, COLS>(g1, (id - n2) % nx1, (id - n2) / nx1, 0, red);
}

// ------------------------------------------------------------------------------------------ q, k, v of a few tokens
// The product that makes queries, keys and values of up to 16 tokens, with what follows it in the same launch:
// bias, rotation of queries and keys (pairs (d, d + hd / 2), the whole head rotated), queries out in bfloat16,
// keys and values into their cache pages (as rope_kv_write_kernel of elementwise.hip does it from the float
// product; same formulas, same float arithmetic).  A workgroup takes the two tiles of 16 columns that hold the
// partners of 16 pairs of one head: columns head * hd + 16 j .. and the same + hd / 2; grid (heads * hd / 32), the
// waves split k.
struct RopeWriteArgs {
  const int* positions;        // [T]
  const int* seq_of_token;     // [T]
  const int* block_table;
  int bt_stride;
  const float* inv_freq;       // [hd / 2]
  bf16_t* q_out;               // [T][nh * hd]
  bf16_t* k_pool;              // the layer's offset already added; null: keys and values are not written
  bf16_t* v_pool;
  int page_size;
  int64_t page_stride;
  int nh, nkv, hd;
};

__global__ __launch_bounds__(512) void qkv_rope_write_kernel(MfmaGemmArgs g, RopeWriteArgs p) {
  extern __shared__ float red[];       // [waves][2][4][64]
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, nw = blockDim.x / 64;
  const int r = lane % 16, c = lane / 16;
  const int per_head = p.hd / 32;
  const int head = blockIdx.x / per_head, j = blockIdx.x % per_head;
  const int col0[2] = {head * p.hd + 16 * j, head * p.hd + p.hd / 2 + 16 * j};
  const int q = c + 4 * (r / 8);
  const bf16_t* ap[1][2];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    const int m = 8 * hf + r % 8;
    ap[0][hf] = m < g.M ? g.a + (size_t)m * g.lda + q * 8 : nullptr;
  }
  const int steps = (g.K + 31) / 32;
  const int per = ((steps + nw - 1) / nw + 1) & ~1;
  const int k_beg = wave * per * 32, k_end = min(g.K, (wave + 1) * per * 32);
  f32x4 acc[2][1], acc2[1][1];
  stream_accumulate<1, false, 2>(g, col0, 0, ap, q, k_beg, k_end, acc, acc2);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[((wave * 2 + t) * 4 + v) * 64 + lane] = acc[t][0][v];
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += blockDim.x) {
    const int ol = i % 64, v = i / 64;
    const int m = 4 * (ol / 16) + v, d = 16 * j + ol % 16;      // token and dimension (of the pair's first half)
    if (m >= g.M) continue;
    float a = 0.f, b = 0.f;
    for (int w = 0; w < nw; ++w) {      // in wave order, as the product alone adds them
      a += red[((w * 2 + 0) * 4 + v) * 64 + ol];
      b += red[((w * 2 + 1) * 4 + v) * 64 + ol];
    }
    a += bias_at(g, col0[0] + ol % 16);
    b += bias_at(g, col0[1] + ol % 16);
    const int pos = p.positions[m];
    if (head < p.nh + p.nkv) {
      const float theta = (float)pos * p.inv_freq[d];
      float sn, cs;
      sincosf(theta, &sn, &cs);
      const float ra = a * cs - b * sn, rb = a * sn + b * cs;
      a = ra;
      b = rb;
    }
    if (head < p.nh) {
      bf16_t* dst = p.q_out + ((size_t)m * p.nh + head) * p.hd;
      dst[d] = f32_to_bf16(a);
      dst[d + p.hd / 2] = f32_to_bf16(b);
      continue;
    }
    if (!p.k_pool) continue;
    const int page = p.block_table[(size_t)p.seq_of_token[m] * p.bt_stride + pos / p.page_size];
    const int row = pos % p.page_size;
    const size_t kv_head_stride = (size_t)p.page_size * p.hd;
    if (head < p.nh + p.nkv) {         // keys lie [row][hd]
      bf16_t* dst = p.k_pool + (size_t)page * p.page_stride + (size_t)(head - p.nh) * kv_head_stride + (size_t)row * p.hd;
      dst[d] = f32_to_bf16(a);
      dst[d + p.hd / 2] = f32_to_bf16(b);
    } else {                           // values lie transposed, [hd][row]
      bf16_t* dst = p.v_pool + (size_t)page * p.page_stride + (size_t)(head - p.nh - p.nkv) * kv_head_stride + row;
      dst[(size_t)d * p.page_size] = f32_to_bf16(a);
      dst[(size_t)(d + p.hd / 2) * p.page_size] = f32_to_bf16(b);
    }
  }
}

// ------------------------------------------------------------------------------------------ many rows
// grid (row tiles of BM, ceil(N / BN)); block of 8 waves laid WM x WN over the tile of BM x BN outputs (BN = 128
// unless said): BM = 128 as 4 x 2 (a wave owns 32 x 64 outputs, or 32 x 96 with BN = 192; the experts' gated pair as 2
// x 4, 64 x 32 of each of its two products), BM = 256 as 4 x 2 (64 x 64 or 64 x 96), BM = 64 as 2 x 4 (32 x 32).
// Eight waves beat four here: twice the waves hide twice the latency.
#define TBN 128
// Most LDS for the sums of the waves that split k: 128 KB lets the gated pair of 64 rows have 8 waves (22.7 us for the
// shared expert at 64 rows against 25.1 with 4).
#define TQ_STREAM_LDS (128 * 1024)

// Where 16-byte chunk `chunk` of row `row` lies in a tile: rows of 128 bytes, the chunk index XOR-ed with bits 1..3
// of the row.  Measured with ds_read_b128 in the operand layout (lane l reads row l % 32): this runs at the full
// 128 bytes per clock; XOR with bits 0..2 at 107, no swizzle at 31.
__device__ __forceinline__ int swz(int row, int chunk) { return row * TBK + ((chunk ^ ((row >> 1) & 7)) << 3); }

template <int BM, int WM, int WN, bool DUAL, bool OUT_ACT, int BN = TBN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_tile_kernel(MfmaGemmArgs g) {
  constexpr int NT = 64 * WM * WN;
  constexpr int MI = BM / WM / 32;               // 32-high row tiles per wave
  constexpr int NI = BN / WN / 32;              // 32-wide column tiles per wave
  constexpr int A_CH = BM * 8 / NT;              // 16-byte chunks of the a tile per thread
  constexpr int W_CH = BN * 8 / NT;
  static_assert(MI >= 1 && NI >= 1 && A_CH >= 1 && W_CH >= 1 && BM * 8 % NT == 0 && BN * 8 % NT == 0, "tile layout");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // two buffers, each a tile of `a`, one of `w` and (gated pair) one of `w2`
  constexpr int BUF = (BM + BN * (DUAL ? 2 : 1)) * TBK;
  bf16_t* As = (bf16_t*)smem;
  bf16_t* Ws = As + BM * TBK;
  bf16_t* Vs = Ws + BN * TBK;
  // Which tile this workgroup takes.  Workgroups are dealt to the chip's 8 dies in turn (id % 8), and each die
  // has its own L2: so the tiles are numbered such that one die gets a contiguous run of them.  One matrix: a
  // run goes through bands of 8 row tiles, down a band's column of row tiles first, so that workgroups that run
  // at the same time on a die share their tiles of `a` and of `w` in that die's L2.  A matrix per expert: a run
  // goes expert by expert, so that an expert's matrix is read by one die (by two where a run ends), and within an
  // expert column by column with the expert's row tiles side by side (measured against row tile by row tile: 6 to
  // 12 % faster, the more the more row tiles an expert has); only the row tiles in use are dealt.
  int tile_m, tile_n;
  {
    // an entry of tile_group (and a unit of n_tiles) stands for `ratio` row tiles of this kernel where the row
    // order was padded to a multiple of the tile's height
    const int ratio = g.group_ratio > 1 ? g.group_ratio : 1;
    const int gx = g.tile_group && g.n_tiles ? min(g.n_tiles[0] * ratio, (int)gridDim.x) : (int)gridDim.x;
    const int gy = gridDim.y, total = gx * gy;
    const int id = blockIdx.y * gridDim.x + blockIdx.x;
    const int die = id % 8, q = total / 8, rem = total % 8;
    if (id / 8 >= q + (die < rem ? 1 : 0)) return;
    const int logical = die * q + min(die, rem) + id / 8;
    if (g.tile_group) {
      // the expert whose row tiles [lo, hi) hold row tile logical / gy; within it column by column, the expert's
      // row tiles of a column one after the other, so that they read that column's rows of w at the same time
      const int u = logical / gy / ratio, e = g.tile_group[u], gu = gx / ratio;
      int lo = u, hi = u + 1;
      while (lo > 0 && g.tile_group[lo - 1] == e) --lo;
      while (hi < gu && g.tile_group[hi] == e) ++hi;
      lo *= ratio;
      hi *= ratio;
      const int local = logical - lo * gy, n_e = hi - lo;
      tile_n = local / n_e;
      tile_m = lo + local % n_e;
    } else {
      const int band = logical / (8 * gy), in_band = logical % (8 * gy);
      const int bh = min(8, gx - band * 8);
      tile_m = band * 8 + in_band % bh;
      tile_n = in_band / bh;
    }
  }
  const int group = g.tile_group ? g.tile_group[tile_m / (g.group_ratio > 1 ? g.group_ratio : 1)] : 0;
  const bf16_t* w = g.w + (size_t)group * g.group_stride;
  const bf16_t* w2 = DUAL ? g.w2 + (size_t)group * g.group_stride : nullptr;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  // an expert's rows stand at the head of its units: a tile that begins with a row of padding holds nothing else
  if (g.tile_group && g.a_rows && g.a_rows[min(m0, g.M - 1)] < 0) return;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / WN, wn = wave % WN;
  // A wave whose rows of an expert's tile are all padding (the expert's last tile is half empty on average) has
  // nothing to multiply: it fetches and stages its share of the tile and waits at the barriers.
  const int wave_m0 = m0 + wm * (MI * 32);
  const bool active = !(g.tile_group && g.a_rows) || (wave_m0 < g.M && g.a_rows[wave_m0] >= 0);
  // this workgroup's run of k: k_lo .. k_lo + Kl (all of k unless the product is split), and where its sums go
  const int k_lo = blockIdx.z * g.k_per;
  const int Kl = min(g.K, k_lo + g.k_per) - k_lo;
  if (blockIdx.z) {
    g.out = (float*)g.out + blockIdx.z * g.split_stride;
    g.bias = nullptr;
  }

  // What this thread fetches of each tile: chunk `ch` of row `row`.  Rows past the end of `a` or `w`, and rows
  // of padding in an expert's tile, read some valid row instead: an output depends on its own row of `a` and
  // of `w` only, and those outputs are never stored.  So the loads need no predicate.
  const bf16_t* a_src[A_CH];
  int a_dst[A_CH], w_dst[W_CH];
  const bf16_t *w_src[W_CH], *v_src[W_CH];
#pragma unroll
  for (int i = 0; i < A_CH; ++i) {
    const int idx = tid + i * NT, row = idx / 8, ch = idx % 8;
    const int m = min(m0 + row, g.M - 1);
    int src = m;
    if (g.a_rows && g.a_gather) src = max(g.a_rows[m], 0);
    a_src[i] = g.a + (size_t)src * g.lda + k_lo + ch * 8;
    a_dst[i] = swz(row, ch);
  }
#pragma unroll
  for (int i = 0; i < W_CH; ++i) {
    const int idx = tid + i * NT, row = idx / 8, ch = idx % 8;
    const int n = min(n0 + row, g.N - 1);
    w_src[i] = w + (size_t)n * g.K + k_lo + ch * 8;
    v_src[i] = DUAL ? w2 + (size_t)n * g.K + k_lo + ch * 8 : nullptr;
    w_dst[i] = swz(row, ch);
  }
  const int ch_of_thread = tid % 8;     // (tid + i * NT) % 8

  f32x16 acc[MI][NI], acc2[DUAL ? MI : 1][DUAL ? NI : 1];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[mi][ni][v] = 0.f;
        if (DUAL) acc2[mi][ni][v] = 0.f;
      }

  u32x4 pa[A_CH], pw[W_CH], pv[DUAL ? W_CH : 1];
  const u32x4 z = {0u, 0u, 0u, 0u};
  // FETCH: the thread's chunks of the tile at k0 into registers; only the last tile of a K that is no multiple
  // of 64 needs zeros past the end.  STAGE: registers into LDS.  (Written as macros so that the small arrays
  // above are only ever indexed by constants and stay in registers.)
#define TQ_FETCH(k0)                                                                                          \
  do {                                                                                                        \
    if ((k0) + TBK <= Kl) {                                                                                   \
      _Pragma("unroll") for (int i = 0; i < A_CH; ++i)                                                        \
          pa[i] = *reinterpret_cast<const u32x4*>(a_src[i] + (k0));                                           \
      _Pragma("unroll") for (int i = 0; i < W_CH; ++i) {                                                      \
        pw[i] = *reinterpret_cast<const u32x4*>(w_src[i] + (k0));                                             \
        if (DUAL) pv[i] = *reinterpret_cast<const u32x4*>(v_src[i] + (k0));                                   \
      }                                                                                                       \
    } else {                                                                                                  \
      const bool k_ok = (k0) + ch_of_thread * 8 < Kl;                                                         \
      _Pragma("unroll") for (int i = 0; i < A_CH; ++i)                                                        \
          pa[i] = k_ok ? *reinterpret_cast<const u32x4*>(a_src[i] + (k0)) : z;                                \
      _Pragma("unroll") for (int i = 0; i < W_CH; ++i) {                                                      \
        pw[i] = k_ok ? *reinterpret_cast<const u32x4*>(w_src[i] + (k0)) : z;                                  \
        if (DUAL) pv[i] = k_ok ? *reinterpret_cast<const u32x4*>(v_src[i] + (k0)) : z;                        \
      }                                                                                                       \
    }                                                                                                         \
  } while (0)
#define TQ_STAGE(off)                                                                                         \
  do {                                                                                                        \
    _Pragma("unroll") for (int i = 0; i < A_CH; ++i) *reinterpret_cast<u32x4*>(As + (off) + a_dst[i]) = pa[i]; \
    _Pragma("unroll") for (int i = 0; i < W_CH; ++i) {                                                        \
      *reinterpret_cast<u32x4*>(Ws + (off) + w_dst[i]) = pw[i];                                               \
      if (DUAL) *reinterpret_cast<u32x4*>(Vs + (off) + w_dst[i]) = pv[i];                                     \
    }                                                                                                         \
  } while (0)

  // Tile t is computed from buffer t % 2 while tile t + 1 goes from registers into the other buffer and tile
  // t + 2 is on its way from memory into registers: one barrier per step of 64 of k.
  TQ_FETCH(0);
  TQ_STAGE(0);
  if (TBK < Kl) TQ_FETCH(TBK);
  __syncthreads();
  const int lr = lane % 32, lc = lane / 32;
  int cur = 0;
  for (int k0 = 0; k0 < Kl; k0 += TBK, cur ^= BUF) {
    if (k0 + TBK < Kl) {
      TQ_STAGE(cur ^ BUF);
      if (k0 + 2 * TBK < Kl) TQ_FETCH(k0 + 2 * TBK);
    }
    const bf16_t* Ac = As + cur;
    const bf16_t* Wc = Ws + cur;
    const bf16_t* Vc = Vs + cur;
    if (active)
#pragma unroll
    for (int j = 0; j < TBK / 16; ++j) {
      bf16x8 af[MI], wf[NI], vf[DUAL ? NI : 1];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const int row = wm * (MI * 32) + mi * 32 + lr;
        af[mi] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(Ac + swz(row, 2 * j + lc)));
      }
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) {
        const int row = wn * (NI * 32) + ni * 32 + lr;
        wf[ni] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(Wc + swz(row, 2 * j + lc)));
        if (DUAL) vf[ni] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(Vc + swz(row, 2 * j + lc)));
      }
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[mi], wf[ni], acc[mi][ni], 0, 0, 0);
          if (DUAL) acc2[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[mi], vf[ni], acc2[mi][ni], 0, 0, 0);
        }
    }
    __syncthreads();
  }
#undef TQ_FETCH
#undef TQ_STAGE

  if (!active) return;
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int n = n0 + wn * (NI * 32) + ni * 32 + lr;
    if (n >= g.N) continue;
    const float b = bias_at(g, n);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm * (MI * 32) + mi * 32 + 8 * (v / 4) + 4 * lc + (v % 4);
        if (m >= g.M) continue;
        if (g.a_rows && g.a_rows[m] < 0) continue;
        float o = acc[mi][ni][v] + b;
        if (DUAL) o = gated_pair(o, acc2[mi][ni][v], g.gate, g.limit);
        store_out<OUT_ACT>(g, m, n, o);
      }
  }
}

// ------------------------------------------------------------------------------------------ a few hundred rows, one matrix
// Tiles of 64 x 32 WN outputs by 2 x WN waves of 32 x 32 each (of either matrix of a gated pair), 64 of k at a time.
// Such a product has a workgroup or two per compute unit, and its time is the steps of one of them: the tile kernel
// takes 0.8 us a step here (load, wait, store into LDS, barrier, and every product behind its own reads), for 64 x 128
// outputs, so that 97 rows by 6,144 x 2,048 kept 96 compute units busy for 26 us.  Here the tiles are smaller where
// that fills the chip, go from memory straight into a ring of S stages of LDS, S - 1 of them on their way while one is
// multiplied (global_load_lds_dwordx4: no registers in between; a load instruction of a wave fills eight rows of 128 bytes, lane l
// the l-th chunk of 16, so the swizzle is in what a lane asks for): 15.0 us, 0.4 us a step.  Two tiles of 64 to a step: 15.9.  The compiler puts a
// step's products between its reads of LDS; all reads before the first product, held there by a scheduling barrier, is
// level (14.8; a gated pair of 97 rows by twice 5,632 x 2,048 23.6 and 23.6, by twice 20,480 x 3,584 85.9 and 85.2, of
// 512 rows by that 229 and 240, of 320 161 and 159).  The sums of an output run over k as in the tile kernel: same bits.
template <int WN, bool DUAL, bool OUT_ACT, int S>
__global__ __launch_bounds__(128 * WN) void gemm_few_tiles_kernel(MfmaGemmArgs g) {
  constexpr int NT = 128 * WN, BM = 64, BN = 32 * WN, ROWS = BM + BN * (DUAL ? 2 : 1), STAGE = ROWS * TBK, L = ROWS * 8 / NT;
  static_assert(ROWS * 8 % NT == 0 && (S - 2) * L < 16 && S >= 2, "ring");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* ring = (bf16_t*)smem;
  // a die gets a contiguous run of tiles, a column's row tiles one after the other
  int tile_m, tile_n;
  {
    const int gx = gridDim.x, total = gx * gridDim.y, id = blockIdx.y * gx + blockIdx.x;
    const int die = id % 8, q = total / 8, rem = total % 8;
    const int logical = die * q + min(die, rem) + id / 8;
    tile_m = logical % gx;
    tile_n = logical / gx;
  }
  const int k_lo = blockIdx.z * g.k_per, steps = (min(g.K, k_lo + g.k_per) - k_lo) / TBK;
  if (blockIdx.z) {
    g.out = (float*)g.out + blockIdx.z * g.split_stride;
    g.bias = nullptr;
  }
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / WN, wn = wave % WN;
  // What this thread asks for of each stage: the chunk that belongs at place tid % 8 of rows tid / 8 + i NT / 8.  Rows past the
  // end read the last row instead: those outputs are never stored.
  const bf16_t* src[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int row = tid / 8 + i * (NT / 8), chunk = (tid % 8) ^ ((row >> 1) & 7);
    const bf16_t* from = row < BM        ? g.a + (size_t)min(m0 + row, g.M - 1) * g.lda
                         : row < BM + BN ? g.w + (size_t)min(n0 + row - BM, g.N - 1) * g.K
                                         : g.w2 + (size_t)min(n0 + row - BM - BN, g.N - 1) * g.K;
    src[i] = from + k_lo + chunk * 8;
  }
  auto issue = [&](int stage, int step) {
#pragma unroll
    for (int i = 0; i < L; ++i) load_to_lds16(src[i] + step * TBK, ring + stage * STAGE + (i * (NT / 8) + wave * 8) * TBK);
  };
  f32x16 acc, acc2;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f, acc2[v] = 0.f;
  for (int s = 0; s < S - 1 && s < steps; ++s) issue(s, s);
  const int lr = lane % 32, lc = lane / 32;
  int cur = 0;
  for (int t = 0; t < steps; ++t) {
    // tile t is in LDS once no more loads of this wave are on their way than those of the tiles behind it, and its reads of tile
    // t - 1 have come back, wherever their products stand
    if (steps - 1 - t >= S - 2)
      __builtin_amdgcn_s_waitcnt(0x0070 | (S - 2) * L);
    else
      __builtin_amdgcn_s_waitcnt(0x0070);
    // every wave's share of tile t has landed and every wave is through with tile t - 1, whose stage tile t + S - 1 takes
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + S - 1 < steps) {
      int nxt = cur + S - 1;
      if (nxt >= S) nxt -= S;
      issue(nxt, t + S - 1);
    }
    const bf16_t* Ac = ring + cur * STAGE;
    const bf16_t* Wc = Ac + BM * TBK;
    const bf16_t* Vc = Wc + BN * TBK;
    u32x4 af[TBK / 16], wf[TBK / 16], vf[TBK / 16];
#pragma unroll
    for (int j = 0; j < TBK / 16; ++j) {
      af[j] = *reinterpret_cast<const u32x4*>(Ac + swz(wm * 32 + lr, 2 * j + lc));
      wf[j] = *reinterpret_cast<const u32x4*>(Wc + swz(wn * 32 + lr, 2 * j + lc));
      if (DUAL) vf[j] = *reinterpret_cast<const u32x4*>(Vc + swz(wn * 32 + lr, 2 * j + lc));
    }
#pragma unroll
    for (int j = 0; j < TBK / 16; ++j) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[j]), __builtin_bit_cast(bf16x8, wf[j]), acc, 0, 0, 0);
      if (DUAL)
        acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[j]), __builtin_bit_cast(bf16x8, vf[j]), acc2, 0, 0, 0);
    }
    if (++cur == S) cur = 0;
  }
  const int n = n0 + wn * 32 + lr;
  if (n >= g.N) return;
  const float b = bias_at(g, n);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = m0 + wm * 32 + 8 * (v / 4) + 4 * lc + (v % 4);
    if (m >= g.M) continue;
    store_out<OUT_ACT>(g, m, n, DUAL ? gated_pair(acc[v] + b, acc2[v], g.gate, g.limit) : acc[v] + b);
  }
}

// ------------------------------------------------------------------------------------------ launch
// Waves that split k in the streaming kernel: a power of two, enough for about 2048 waves on the chip when one
// matrix is multiplied and for about 256 per matrix when there is one per expert, each wave keeping at least 256 of
// k.  A function of N, K and of whether the product is over experts, never of the number of rows.
static int split_k_waves(int N, int K, bool grouped) {
  const int n_tiles = (N + 15) / 16;
  const int want = grouped ? 256 : 2048;
  int s = 1;
  while (s < 16 && n_tiles * s < want && K / (s * 2) >= 256) s *= 2;
  return s;
}

// Whether lean_body takes a product of at most 16 rows a tile.
static bool lean_suits(const MfmaGemmArgs& g) {
  return g.K % 64 == 0 && g.N % 16 == 0 && g.K < (1 << 26) && g.k_per % 64 == 0 &&
         (g.tile_group ? g.a_rows && g.n_tiles : !g.a_rows && !g.n_tiles && g.M <= 16);
}
// A workgroup's columns there.  Tiles of 8 leave fewer compute units without work but read `a` twice as often, which costs the more
// the more rows there are and the less `w` has of them (a gated pair reads two lines of w for one of a).
// One matrix: 8 where tiles of 16 do not give three quarters of the compute units one (one row by 2,048 x 5,632: 6.9 us against 8.7 in
// tiles of 16; sixteen 10.8 and 13.3; from five eighths on for up to 8 rows: sixteen by 2,816 x 1,024 5.5 and 4.7), and where they
// come out unevenly for up to 8 rows, 12 of a gated pair (384 tiles, one row by 6,144 x 2,048 7.3 and 8.0; eight of a pair 12.9 and
// 13.8); else few rows of wide matrices alone (one row by 20,480 x 3,584 24.6 and 26.0, four of a pair 48.5 and 50.4; of a pair by
// 8,192 x 4,096 25.6 and 23.8; eight rows by 151,936 x 2,048 144 and 116, sixteen of a pair by 11,008 x 4,096 47.7 and 37.1).
// A matrix per expert: while row tiles are few (60 experts of 1,408 x 2,048, four a token, us of the pair and of the second product: one
// token 9.7 7.2 and 11.2 7.1, four 27.8 17.0 and 27.6 14.7, sixteen 69.8 36.9 and 66.4 34.5, 64 109 65 and 108 54; with a second
// product beside them sixteen 70.3 39.8 and 70.3 37.5).
static int lean_columns(const MfmaGemmArgs& g, int row_tiles, bool dual) {
  if (g.tile_group) return row_tiles <= (dual ? 16 : 6) ? 8 : 16;
  const int tiles = g.N / 16, rounds = (tiles + 255) / 256;
  if (tiles <= 256) return tiles < (g.M > 8 ? 160 : 192) ? 8 : 16;
  const bool uneven = rounds * 256 > tiles + tiles / 4;
  return g.M <= (dual ? (uneven ? 12 : tiles > 512 ? 4 : 0) : (uneven ? 8 : 1)) ? 8 : 16;
}

// MT row tiles of 16; more than one (17 to 64 rows of one matrix) go with two column tiles per wave.
template <int MT>
static int launch_stream(MfmaGemmArgs g, bool dual, bool out_act, int row_tiles, hipStream_t st, int splits = 1) {
  constexpr int NTL = MT > 1 ? 2 : 1;
  if (splits > 1) {        // runs of k, each a multiple of 64 so that it starts at a whole line
    g.k_per = ((g.K + 63) / 64 + splits - 1) / splits * 64;
    if ((int64_t)(splits - 1) * g.k_per >= g.K) return TQ_ERR_BAD_ARG;
  }
  int nw = split_k_waves((g.N + NTL - 1) / NTL, splits > 1 ? g.k_per : g.K, g.tile_group != nullptr);
  const size_t per_wave = (size_t)NTL * MT * (dual ? 2 : 1) * 4 * 64 * sizeof(float);
  while (nw > 1 && (nw * per_wave > TQ_STREAM_LDS || (NTL > 1 && nw > 8))) nw /= 2;
  const dim3 grid((g.N + 16 * NTL - 1) / (16 * NTL), row_tiles, splits);
  const size_t shmem = nw > 1 ? nw * per_wave : 0;
  if (shmem > TQ_STREAM_LDS) return TQ_ERR_UNSUPPORTED;
  if constexpr (MT == 1) {
    if (lean_suits(g)) {
      const int cols = lean_columns(g, row_tiles, dual);
      const dim3 lean_grid(g.N / cols, row_tiles, splits);
#define TQ_LEAN(D, O, G, C) hipLaunchKernelGGL((gemm_lean_kernel<D, O, G, C>), lean_grid, dim3(64 * nw), shmem, st, g)
#define TQ_LEAN_OF(D, O)                                            \
  do {                                                              \
    if (g.tile_group && cols == 8) TQ_LEAN(D, O, true, 8);          \
    else if (g.tile_group) TQ_LEAN(D, O, true, 16);                 \
    else if (cols == 8) TQ_LEAN(D, O, false, 8);                    \
    else TQ_LEAN(D, O, false, 16);                                  \
  } while (0)
      if (dual && out_act) TQ_LEAN_OF(true, true);
      else if (dual) TQ_LEAN_OF(true, false);
      else if (out_act) TQ_LEAN_OF(false, true);
      else TQ_LEAN_OF(false, false);
#undef TQ_LEAN_OF
#undef TQ_LEAN
      return 0;
    }
  }
#define TQ_STREAM(D, O)                                                                                       \
  do {                                                                                                        \
    if (shmem > 48 * 1024)                                                                                    \
      (void)hipFuncSetAttribute((const void*)gemm_stream_kernel<MT, D, O, NTL>,                               \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);                      \
    hipLaunchKernelGGL((gemm_stream_kernel<MT, D, O, NTL>), grid, dim3(64 * nw), shmem, st, g);               \
  } while (0)
  if (dual && out_act) TQ_STREAM(true, true);
  else if (dual) TQ_STREAM(true, false);
  else if (out_act) TQ_STREAM(false, true);
  else TQ_STREAM(false, false);
#undef TQ_STREAM
  return 0;
}

template <int BM, int WM, int WN, int BN = TBN>
static int launch_tile(const MfmaGemmArgs& g, bool dual, bool out_act, int splits, hipStream_t st) {
  const dim3 grid((g.M + BM - 1) / BM, (g.N + BN - 1) / BN, splits);
  const size_t shmem = (size_t)2 * (BM + BN * (dual ? 2 : 1)) * TBK * sizeof(bf16_t);
#define TQ_TILE(D, O)                                                                                  \
  do {                                                                                                 \
    if (shmem > 48 * 1024)                                                                             \
      (void)hipFuncSetAttribute((const void*)gemm_tile_kernel<BM, WM, WN, D, O, BN>,                         \
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);                     \
    hipLaunchKernelGGL((gemm_tile_kernel<BM, WM, WN, D, O, BN>), grid, dim3(64 * WM * WN), shmem, st,  \
                       g);                                                                             \
  } while (0)
  if (dual && out_act)
    TQ_TILE(true, true);
  else if (dual)
    TQ_TILE(true, false);
  else if (out_act)
    TQ_TILE(false, true);
  else
    TQ_TILE(false, false);
#undef TQ_TILE
  return 0;
}

template <int WN, int S, bool DUAL>
static int launch_few_tiles(const MfmaGemmArgs& g, bool out_act, int splits, hipStream_t st) {
  const dim3 grid((g.M + 63) / 64, (g.N + 32 * WN - 1) / (32 * WN), splits);
  const size_t shmem = (size_t)S * (64 + 32 * WN * (DUAL ? 2 : 1)) * TBK * sizeof(bf16_t);
  const auto kernel = out_act ? gemm_few_tiles_kernel<WN, DUAL, true, S> : gemm_few_tiles_kernel<WN, DUAL, false, S>;
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
    return TQ_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kernel, grid, dim3(128 * WN), shmem, st, g);
  return 0;
}

// Which of its tiles a product of gemm_few_tiles_kernel takes.  Narrow ones, with a deep ring, while there is at most
// one to a compute unit: then what counts is how soon a tile is done (97 rows by 6,144 x 2,048: 15.0 us against 19.2
// in wide ones and 26.0 in the tile kernel).  More of them take wide tiles, which read `a` half as often (320 rows:
// 20.2 against 22.3, tile kernel 26.1).  A gated pair has two matrices' tiles in a stage and so fewer stages (97 rows
// by twice 5,632 x 2,048: 23.5 us, tile kernel 35.6; 320 rows in wide ones 30.8, 35.7), and where its tiles are many,
// rings of two stages that leave room for three narrow or two wide tiles on a compute unit: 512 rows 47 in narrow
// ones, 57 in wide ones of three stages, 61 in the tile kernel; 320 rows by twice 20,480 x 3,584, more than three
// narrow ones to a unit: 157 in wide ones, 176 in narrow ones, tile kernel 174.
static int launch_few_tiles(const MfmaGemmArgs& g, bool dual, bool out_act, int splits, hipStream_t st) {
  const int64_t narrow = (int64_t)((g.M + 63) / 64) * ((g.N + 63) / 64) * splits;
  if (!dual) return narrow <= 256 ? launch_few_tiles<2, 4, false>(g, out_act, splits, st) : launch_few_tiles<4, 3, false>(g, out_act, splits, st);
  if (narrow <= 256) return launch_few_tiles<2, 3, true>(g, out_act, splits, st);
  if (narrow <= 512) return launch_few_tiles<4, 3, true>(g, out_act, splits, st);
  if (narrow <= 768) return launch_few_tiles<2, 2, true>(g, out_act, splits, st);
  return launch_few_tiles<4, 2, true>(g, out_act, splits, st);
}

// Whether a product of 17 to 64 rows takes the tiled kernel: a matrix wide enough to give every compute unit two
// tiles of 128 columns (a vocabulary).  The tiles read `a` through LDS once per 128 columns, the streaming kernel
// once per 32 (measured at 151,936 x 2,048 and 64 rows: 159 us against 466 with 16 columns a wave).
static bool wide_enough_for_tiles(int N) { return (N + TBN - 1) / TBN >= 512 && (N + TBN - 1) / TBN <= 65535; }

// Whether a product in tiles of 64 rows goes to gemm_few_tiles_kernel rather than the tile kernel: rows that follow
// one another, k in whole tiles, and up to 512 rows (512 by 2,048 x 5,632: 26.6 us against 27.8; 768 rows: 39.7
// against 38.0), of a very wide matrix up to 128 (128 by 65,536 x 1,024: 49.7 against 53.1; 512 rows: 160 against
// 151).  A gated pair up to 1,024 (twice 5,632 x 2,048: 86 against 120; 20,480 x 3,584: 422 against 438).
static bool few_tiles_suit(const MfmaGemmArgs& g, bool dual) {
  const int most = dual ? 1024 : wide_enough_for_tiles(g.N) ? 128 : 512;
  return !g.a_rows && g.K % TBK == 0 && g.M <= most;
}

// Which tile a plain product of many rows takes: 128 x 128, 128 x 192, 256 x 128 or 256 x 192 outputs (0..3).  The
// larger the tile, the fewer bytes pass through LDS per multiply-add (measured on products that fill the chip
// evenly: 1.06, 1.05 and 1.12 times the rate of 128 x 128); against that stand the compute units left idle when
// the tiles do not divide evenly among the 256 of them, and the rows and columns of padding at the edges.  2,048
// rows by 6,144 columns are 768, 512, 384 or 256 tiles: three, two, one and a half, or one to a compute unit.
static int plain_tile_choice(int M, int N, int splits) {
  static const int bm[4] = {128, 128, 256, 256}, bn[4] = {128, 192, 128, 192};
  static const double rate[4] = {1.0, 1.06, 1.05, 1.12};
  int best = 0;
  double best_score = 0.0;
  for (int c = 0; c < 4; ++c) {
    const double rows = (M + bm[c] - 1) / bm[c], cols = (N + bn[c] - 1) / bn[c];
    const double per_cu = rows * cols * splits / 256.0;
    const double even = per_cu / (double)(int64_t)(per_cu + 0.999999);
    const double useful = ((double)M * N) / (rows * bm[c] * cols * bn[c]);
    const double score = rate[c] * even * useful;
    if (score > best_score * 1.0001) {
      best = c;
      best_score = score;
    }
  }
  return best;
}

// Whether a gated pair of a few hundred rows with one matrix goes in tiles of 64 rows rather than 128.  With so few
// rows a workgroup's time is its steps over k, 1.0 us a step in the lower tile against 1.35 in the taller, as long as
// it has its compute unit to itself; of the lower tiles two fit on a compute unit (80 KB of LDS each), of the
// taller one.  So: the lower tile where it needs no more than one workgroup to a compute unit, or where the
// taller one would need a second round and the lower fits in one (320 rows by 2 x 5,632 x 2,048: 34 us against
// 46; 384 rows: 47 against 46; 192 rows by 2 x 20,480 x 3,584: 103 against 149; 128 rows: 110 against 92).
static bool gated_pair_in_tiles_of_64(int M, int N) {
  const int64_t cols = (N + TBN - 1) / TBN;
  const int64_t lower = (int64_t)((M + 63) / 64) * cols, taller = (int64_t)((M + 127) / 128) * cols;
  return lower <= 256 || (taller > 256 && lower <= 512);
}

// How long gemm_phases takes for a product of one matrix in tiles of 64 mi rows, k in runs, us: 8 in front of and behind a tile's steps
// of 64, and a step's time, which grows with how many compute units are at work beside it (the clock falls with the power they draw):
// the first figure where few are, the second where all are.  Fitted to 1,400 timings (80 to 13,197 rows, 64 to 151,936 columns, k 1,024 to
// 20,480): 4 % above them on average, 9 % off in the root of the mean square, and the height it names loses 0.1 % to the best one.
static double phases_time(int M, int N, int K, bool dual, int mi, int runs) {
  static const double few[5] = {0, 0.50, 0.62, 0.84, 1.10}, all[5] = {0, 0.60, 0.86, 1.10, 1.48};
  const int cols = dual ? 128 : 256, steps = (K / TBK + runs - 1) / runs;
  const int64_t tiles = (int64_t)((M + 64 * mi - 1) / (64 * mi)) * ((N + cols - 1) / cols) * runs;
  const double busy = (double)(tiles % 256) / 256;
  return (double)(tiles / 256) * (8 + all[mi] * steps) + (busy > 0 ? 8 + steps * (few[mi] + (all[mi] - few[mi]) * busy) : 0);
}
static double phases_best(int M, int N, int K, bool dual, int runs, int* rows) {
  double best = 0;
  for (int mi = 1; mi <= 4 && (mi == 1 || M > 64 * (mi - 1)); ++mi) {
    const double t = phases_time(M, N, K, dual, mi, runs);
    if (mi == 1 || t < best) best = t, *rows = 64 * mi;
  }
  return best;
}

// Runs of k in the tile kernel where partial sums are wanted apart (see tq_gemm_mfma_splits).
static int tile_kernel_runs(int M, int N, int K) {
  const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + TBN - 1) / TBN);
  int s = 1;
  while (s < 4 && tiles * s < 512 && K / (s * 2) >= 1024) s *= 2;
  return s;
}

// Whether a product of one matrix, of more than 64 rows that follow one another, goes in the tiles of gemm_phases rather than those of
// gemm_few_tiles or the tile kernel: k in whole tiles, and
//  * more than 1,024 rows: always (us by the tile kernel and by gemm_phases: 1,280 rows by 2,048 x 2,048 31.8 and 25.3, 3,001 by 3,072 x
//    2,048 84.6 and 44.5, 13,197 by 6,144 x 2,048 424 and 271; gated pairs of 2,048 rows by 5,632 x 2,048 186 and 88);
//  * 513 to 1,024 where tiles of 64 x 128 do not find a compute unit each (264 of them, 700 by 3,072 x 2,048, 29.5 and 25.5; 176,
//    700 by 2,048 x 5,632, 45.6 and 53.1) and a tile has some steps (741 by 6,464 x 128 11.1 and 13.1);
//  * up to 512 where there are more than two of them to a unit (528, 512 by 8,448 x 2,048, 39.0 and 29.6; 512, 200 by 16,384 x 2,048,
//    26.8 and 26.2; 384, 512 by 6,144 x 2,048, 25.2 and 26.6; 256, 128 by 16,384 x 2,048, 17.9 and 24.7);
//  * a gated pair of up to 1,024 where tiles of 64 x 64 do not find a unit each (264, 160 by 5,632 x 2,048, 27.1 and 23.9; 220, 320 by
//    2,816 x 1,024, 16.1 and 16.0; 160, 256 by 2,560 x 3,584, 32.5 and 34.7).
// And columns in whole pieces of 16 bytes of the result: without, a lane's four or eight columns side by side go out one by one (10,405
// by 314 x 320 15.3 and 20.2, 4,377 by 5,006 x 2,752 141 and 162, 727 by 5,583 x 448 15.8 and 22.8).
// Up to 32 columns are an eighth of these tiles, and a quarter of the tile kernel's: plain products of those only with k long enough,
// rows that are one round of tiles of 64, and no partial sums apart (by 16 columns, us by the tile kernel and by gemm_phases: 4,096 x 512
// 11.2 and 12.5, 4,096 x 2,048 20.1 and 18.4, 28,000 x 2,048 25.6 and 28.4; apart 16,384 x 2,048 15.8 and 23.1, 8,192 x 4,096 18.2 and
// 21.3; a gated pair gains everywhere).  Partial sums of up to 128 columns, half of these tiles, stay where the tile kernel's runs are
// just one round of its tiles (14,000 by 40 x 2,048 19.0 and 21.4, 16,384 by 64 x 2,048 21.6 and 25.8).  runs: of k, 1 where they are not apart.
static bool phases_suit(int M, int N, int K, bool dual, int runs) {
  if (M <= 64 || K % TBK || K < 2 * TBK || N % 8) return false;
  if (!dual && N <= 32 && (runs > 1 || K < 2048 || M > 64 * 256)) return false;
  const int round = (M + 127) / 128 * runs;
  if (runs > 1 && N <= 128 && runs == tile_kernel_runs(M, N, K) && round >= 200 && round <= 256) return false;
  const int64_t rows = (M + 63) / 64, narrow = rows * ((N + 63) / 64), wide = rows * ((N + 127) / 128);
  if (M > 1024) return true;
  return dual ? narrow > 256 : wide > (M > 512 ? 256 : 512) && K >= 512;
}
// The height of those tiles for a product of one matrix whose rows follow one another (dual: a gated pair), k in `splits` runs; 0: it goes in others.
TQ_API int tq_gemm_phases_rows(int M, int N, int K, int dual, int splits) {
  if (!phases_suit(M, N, K, dual != 0, splits)) return 0;
  int rows;
  phases_best(M, N, K, dual != 0, splits, &rows);
  return rows;
}
// Its runs of k where partial sums are wanted apart, `from` at least (the tile kernel's: fewer runs are longer sums, whose error against
// 64 bits is the larger, 2.7e-7 of 2,048 products in one run and 1.9e-7 in two): what a run more saves must be more than writing and
// reading its sums takes, and they stay within 256 MB, which the kernel behind reads.
static int phases_runs(int M, int N, int K, int from) {
  int best = from, rows;
  double least = phases_best(M, N, K, false, from, &rows) + (from - 1) * ((double)M * N * 8 / 5e6);
  for (int s = 2 * from; s <= 4 && (int64_t)s * M * N * 4 <= (256 << 20); s *= 2) {
    const int per = (K / TBK + s - 1) / s;
    if (per < 4 || K / TBK - per * (s - 1) < 2) break;
    const double t = phases_best(M, N, K, false, s, &rows) + (s - 1) * ((double)M * N * 8 / 5e6);
    if (t < least) least = t, best = s;
  }
  return best;
}

TQ_API int tq_gemm_mfma_splits(int M, int N, int K);

// Whether a product of many rows that the vendor's library would take is the faster one here.  kind 0: plain; 1: its result passes an
// activation alone; 2: a gated pair, both into the activation type. The library's kernels leave their sums in float for a pass of its
// own to apply the activation, so that against them stand 14 us (11.5 of an activation alone), the multiply-adds at 1,150 TFLOP/s and
// that pass at 5.5 TB/s (us by the library and here: gated 2,048 by 5,632 x 2,048 105 and 88, 1,999 by 11,008 x 4,096 408 and 288,
// 1,280 by 768 x 1,024 18 and 16, 900 by 1,024 x 4,096 31 and 40; an activation alone 3,001 by 8,448 x 2,048 127 and 103, 768 by
// 1,408 x 2,048 19 and 23, 1,315 by 256 x 832 11 and 13).  A plain product the library does at the same rate, but not where its
// columns are no whole number of tiles (2,048 by 6,288 x 2,048 70 and 55, 1,733 by 7,184 x 2,048 62 and 54, 3,258 by 8,224 x 2,048
// 120 and 109; by 8,448 101 and 102): there where the tiles here reach 950 TFLOP/s, and up to k 2,048.  Beyond, the library adds k in parts
// for many a size: the slower kernel (13,197 by 3,584 x 3,584 367 us and 274 here, 8,192 by 3,584 x 20,480 1,305 and 860), but the
// closer to 64 bits (3.45e-7 against 3.68e-7, 8.3e-7 against 9.2e-7; 17 of 66 sizes drawn from k 2,496 to 12,672, by 4 to 11 %), and a
// result in float keeps what is gained.  Up to k 2,304 the error was the same in all of 24.  (A result of 16 bits is off by 1.7e-3.)
// kind 3: plain, and its partial sums are wanted apart.  Two and four runs of k are closer to 64 bits than the library is (2,048 columns,
// k 8,448: 4.0e-7 and 5.8e-7; 1,024 columns in four 2.7e-7 and 5.7e-7).  Here they go from 1,025 rows, 1,024 to 8,191 columns and k 8,192 on where
//  * their tiles are one round, one to a compute unit at most: 1.00 to 1.44 times as fast as the library, with the sum and norm that read them,
//    in all of 84 such sizes (us by the library and here: 3,258 rows by 2,048 x 8,448 118 and 110; 2,421 by 2,080 x 9,472 106 and 104; 1,121 by
//    5,744 x 12,032 171 and 146; 1,787 by 1,344 x 16,192 121 and 86), twice in 3 where the library takes a slower kernel (1,302 by 3,936 x
//    14,912 308 and 141).  Of more rounds and fewer multiply-adds than the next line's, 33 of 37 lose (1,091 by 7,168 x 8,192 129 and 147, 2,713 by 2,944 x
//    12,928 189 and 222, 5,644 by 1,296 x 8,960 137 and 169, 1,152 by 6,656 x 8,384 124 and 145);
//  * or 1.4e11 multiply-adds: for three of four sizes the library takes kernels there that need half as long again and more (3,258 by 5,120 x
//    11,008 577 and 368, 12,032 by 1,536 x 12,992 715 and 442; 1.23 to 1.78 in 40 of 54), else it is level (4,096 by 6,144 x 8,192 373 and 384,
//    x 14,336 600 and 580, 8,636 by 1,904 x 14,208 448 and 448: 0.97 to 1.07).
// (800 rows by 2,048 x 8,448 51 and 63; fewer than 1,024 columns were not timed.)  Up to k 5,632 it is as often the other way round (2,048
// columns, k 5,632: 0.95 to 1.08, k 3,072 0.88 to 0.95).
TQ_API int tq_gemm_here_rather(int M, int N, int K, int kind) {
  const bool dual = kind == 2;
  if (kind == 3) {
    const int runs = M > 1024 && N >= 1024 && N < 8192 && K >= 8192 ? tq_gemm_mfma_splits(M, N, K) : 1;
    if (runs > 1 && phases_suit(M, N, K, false, runs)) {
      int rows;
      phases_best(M, N, K, false, runs, &rows);
      if ((int64_t)((M + rows - 1) / rows) * ((N + 255) / 256) * runs <= 256 || (int64_t)M * N * K >= 140000000000) return 1;
    }
    kind = 0;
  }
  if (!phases_suit(M, N, K, dual, 1)) return 0;
  int rows;
  const double t = phases_best(M, N, K, dual, 1, &rows), flops = 2.0 * M * N * K * (dual ? 2 : 1);
  if (kind) return (dual ? t : 0.95 * t) <= (dual ? 14 : 11.5) + flops / 1.15e9 + (double)M * N * (dual ? 10 : 6) / 5.5e6;
  return K <= 2048 && N % 256 != 0 && flops / (t * 1e6) >= 950;
}

// Into how many runs of k a plain product of M rows may be split when its partial sums are wanted apart.  Many
// rows: a product whose tiles do not fill the chip twice, and that has k enough, goes faster in 2 to 4 runs, each
// at least 1024 long, and up to 1,024 rows as tile_runs says; in the tiles of gemm_phases in as many, or in more and shorter
// ones (256 of k at least) where phases_runs expects them to be faster.  17 to 64 rows of a narrow matrix with a long k in the
// streaming kernel (at most 8 waves over k): as many runs as bring about 4096 waves, each wave keeping 128 of k
// (64 rows by 2,048 x 2,048: 13.4 us in two runs against 15.2 in one; by 2,048 x 5,632: 17.3 in four against 20.7
// in two); from 33 rows on the tile kernel with its runs instead, where it may split k.  1 for up to 16 rows.
// Runs of k for a product that goes in tiles of 64 rows (up to 1,024 rows): a workgroup's time is its steps over k
// (about 0.6 us each in the tile kernel, whatever the memory does), so up to 8 runs, each at least 256 long, while the workgroups stay
// within two to a compute unit and the partial sums within 8 MB, which the kernel behind has to read (128 rows by
// 2,048 x 2,048: 8.7 us in eight runs against 14.6 in two; by 2,048 x 5,632: 13.7 against 19.3 in four; in the smaller
// tiles of gemm_few_tiles_kernel the eight runs take 7.9 and 12.3).
static int tile_runs(int M, int N, int K) {
  const int64_t tiles64 = (int64_t)((M + 63) / 64) * ((N + TBN - 1) / TBN);
  int t = 1;
  while (t < 8 && tiles64 * t * 2 <= 512 && K / (t * 2) >= 256 && (int64_t)t * 2 * M * N * 4 <= (8 << 20)) t *= 2;
  // every run must begin before the end of k (runs are whole tiles of 64)
  while (t > 1 && (int64_t)(t - 1) * (((K + TBK - 1) / TBK + t - 1) / t * TBK) >= K) t /= 2;
  return t;
}

// Whether partial sums of 33 to 64 rows come from the tile kernel rather than the streaming one: where the tile
// kernel may split k at all.  Its one row tile then has up to eight runs of k to the streaming kernel's two to four
// (64 rows by 2,048 x 2,048: 7.2 us against 13.1; by 2,048 x 5,632: 10.1 against 17.0; by 3,584 x 20,480: 34 against
// 62).
// From 17 to 32 rows it is level (2,048 x 2,048: 6.7 to 7.6 us against 7.8 to 8.7; 2,048 x 5,632: 11.9 to 12.7 against
// 10.6 to 11.8), and the streaming kernel's fewer runs are less for the next kernel to add.
static bool few_rows_in_tiles(int M, int N, int K) {
  return M > 32 && M <= 64 && !wide_enough_for_tiles(N) && tile_runs(M, N, K) > 1;
}

TQ_API int tq_gemm_mfma_splits(int M, int N, int K) {
  if (M <= 16) return 1;
  if (M <= 64) {
    if (wide_enough_for_tiles(N)) return 1;
    if (few_rows_in_tiles(M, N, K)) return tile_runs(M, N, K);
    const int64_t waves = (int64_t)((N + 31) / 32) * 8;
    int s = 1;
    while (s < 8 && waves * s < 4096 && K / (16 * s) >= 128) s *= 2;
    return s;
  }
  int s = tile_kernel_runs(M, N, K);
  if (phases_suit(M, N, K, false, s)) return phases_runs(M, N, K, s);
  if (M <= 64 * 16) {      // tiles of 64 rows: more and shorter runs
    const int t = tile_runs(M, N, K);
    if (t > s) s = t;
  }
  return s;
}

// The queue that tile_rows names, or null, and tile_rows without it; false: what cannot be.  Without a tile_group it is a hint, whatever it says.
static bool take_queue(int& tile_rows, const int* tile_group, const int* n_tiles, int** queue) {
  const int which = tile_rows / TQ_TILE_QUEUE;
  *queue = nullptr;
  if (!tile_group || tile_rows < TQ_TILE_QUEUE) return true;
  tile_rows %= TQ_TILE_QUEUE;
  *queue = const_cast<int*>(n_tiles) + 16 * which;
  return which <= 2 && n_tiles && tile_rows == 64 + TQ_TILE_PAIRS;
}

// a: bfloat16 [.., K] with row stride lda (a multiple of 8, as K must be); w, w2: bfloat16.
// tile_rows: with tile_group set, the padding unit of the row order (16, 32, 64, 128 or 256); else a hint that is
// ignored.  64 + TQ_TILE_PAIRS: units of 64 taken two or four at a time, by the items that the row order lists behind its
// row tiles (tile_group[M / 64 ..], n_tiles[1]); with TQ_TILE_QUEUE once or twice on top, dealt from the order's first or second queue.
// splits > 1 (as tq_gemm_mfma_splits says, for a plain product into float): run z of k goes to out + z * M * ldc,
// the bias to run 0; the sum over the runs is the caller's.
// gate: the activation of the gated pair; without w2 and with TQ_GEMM_ACT_ALONE added, the activation that the plain
// product's result (bias included) passes before it is stored (a feed-forward of two matrices needs no launch between them).
TQ_API int tq_gemm_mfma(const void* a, int64_t lda, const int* a_rows, int a_gather, const void* w, const void* w2,
                        int64_t group_stride, const int* tile_group, const int* n_tiles, const void* bias,
                        int bias_type, void* out, int64_t ldc, int out_is_act, int M, int N, int K, int tile_rows,
                        int splits, int gate, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 8 != 0 || lda % 8 != 0) return TQ_ERR_BAD_ARG;
  if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)w2) % 16 != 0 || (group_stride % 8) != 0) return TQ_ERR_BAD_ARG;
  const bool dual = w2 != nullptr, out_act = out_is_act != 0;
  const bool alone = gate >= TQ_GEMM_ACT_ALONE;
  if (alone) gate -= TQ_GEMM_ACT_ALONE;
  if (splits < 1 || splits > 64 || gate < 0 || gate >= TQ_GATE_COUNT) return TQ_ERR_BAD_ARG;
  if (alone && (dual || splits > 1)) return TQ_ERR_BAD_ARG;
  if (splits > 1 && (dual || out_act || tile_group || a_rows || splits != tq_gemm_mfma_splits(M, N, K))) return TQ_ERR_BAD_ARG;
  const int k_per = ((K + TBK - 1) / TBK + splits - 1) / splits * TBK;
  if (splits > 1 && (int64_t)(splits - 1) * k_per >= K) return TQ_ERR_BAD_ARG;
  int* queue;
  if (!take_queue(tile_rows, tile_group, n_tiles, &queue)) return TQ_ERR_BAD_ARG;
  MfmaGemmArgs g{(const bf16_t*)a, lda, a_rows, a_gather, (const bf16_t*)w, (const bf16_t*)w2, group_stride,
                 tile_group, n_tiles, bias, bias_type, out, ldc, M, N, K, splits > 1 ? k_per : K, (int64_t)M * ldc, gate, 1,
                 alone ? gate + 1 : 0, tq_pair_limit_host};
  int rc = 0;
  if (tile_group) {
    if (tile_rows == 16) {
      if (M % 16) return TQ_ERR_BAD_ARG;
      rc = launch_stream<1>(g, dual, out_act, M / 16, st);
    } else if (tile_rows == 32) {      // the streaming kernel with two row tiles and two column tiles to a wave
      if (M % 32) return TQ_ERR_BAD_ARG;
      rc = launch_stream<2>(g, dual, out_act, M / 32, st);
    } else if (tile_rows == 64 || tile_rows == 64 + TQ_TILE_PAIRS) {
      if ((N + TBN - 1) / TBN > 65535 || M % 64) return TQ_ERR_UNSUPPORTED;
      if (tile_rows != 64 && K % TBK == 0 && K >= 2 * TBK)
        rc = launch_gemm_phases(g, nullptr, queue, dual, out_act, st);
      else
        rc = launch_tile<64, 2, 4>(g, dual, out_act, 1, st);
    } else if (tile_rows == 128) {     // experts with hundreds of rows each: the taller tile's rate for little padding
      if ((N + TBN - 1) / TBN > 65535 || M % 128) return TQ_ERR_UNSUPPORTED;
      // the gated pair as 2 x 4 waves of 64 x 32 outputs (and as many of w2): 3 to 4 % faster than 4 x 2 of 32 x 64
      if (dual)
        rc = launch_tile<128, 2, 4>(g, dual, out_act, 1, st);
      else
        rc = launch_tile<128, 4, 2>(g, dual, out_act, 1, st);
    } else if (tile_rows == 256) {
      // A thousand rows and more each.  The gated pair takes tiles as tall as the unit, a wave's 64 x 64 outputs per
      // pass over its operands (13,199 tokens x 8 of 64 experts of 2,560 x 3,584: 4.37 ms against 5.09 in tiles of 128
      // rows); the plain product, whose k is the shorter one, stays with two tiles of 128 to a unit (2.85 ms; 3.00 as
      // tiles of 256), of which one that holds padding only ends at once.
      if ((N + TBN - 1) / TBN > 65535 || M % 256) return TQ_ERR_UNSUPPORTED;
      if (dual) {
        rc = launch_tile<256, 4, 2>(g, dual, out_act, 1, st);
      } else {
        g.group_ratio = 2;
        rc = launch_tile<128, 4, 2>(g, dual, out_act, 1, st);
      }
    } else {
      return TQ_ERR_BAD_ARG;
    }
  } else if (M <= 16) {
    rc = launch_stream<1>(g, dual, out_act, 1, st);
  } else if (M <= 64 && (wide_enough_for_tiles(N) || (splits > 1 && few_rows_in_tiles(M, N, K)))) {
    if (few_tiles_suit(g, dual))
      rc = launch_few_tiles(g, dual, out_act, splits, st);
    else
      rc = launch_tile<64, 2, 4>(g, dual, out_act, splits, st);
  } else if (M <= 32) {
    rc = launch_stream<2>(g, dual, out_act, 1, st, splits);
  } else if (M <= 64) {
    rc = launch_stream<4>(g, dual, out_act, 1, st, splits);
  } else {
    if ((N + TBN - 1) / TBN > 65535) return TQ_ERR_UNSUPPORTED;
    if (const int rows = a_rows ? 0 : tq_gemm_phases_rows(M, N, K, dual, splits))
      rc = launch_gemm_phases_plain(g, rows, dual, out_act, st);
    else if (few_tiles_suit(g, dual))
      rc = launch_few_tiles(g, dual, out_act, splits, st);
    else if (M <= 64 * 16 && !dual)
      rc = launch_tile<64, 2, 4>(g, dual, out_act, splits, st);
    else if (dual && gated_pair_in_tiles_of_64(M, N))
      rc = launch_tile<64, 2, 4>(g, dual, out_act, splits, st);
    else if (dual)
      rc = launch_tile<128, 4, 2>(g, dual, out_act, splits, st);
    else
      switch (plain_tile_choice(M, N, splits)) {
        case 1: rc = launch_tile<128, 4, 2, 192>(g, dual, out_act, splits, st); break;
        case 2: rc = launch_tile<256, 4, 2, 128>(g, dual, out_act, splits, st); break;
        case 3: rc = launch_tile<256, 4, 2, 192>(g, dual, out_act, splits, st); break;
        default: rc = launch_tile<128, 4, 2>(g, dual, out_act, splits, st);
      }
  }
  if (rc) return rc;
  TQ_LAUNCH_CHECK();
  return 0;
}

// Into how many runs of k the second product of a pair is split when its partial sums are wanted apart: the
// workgroups of a pair have the waves that suit the first product, so a second product that alone would have s
// times as many waves over its k gets s runs instead.  A function of the two products' N and K and of whether each
// has a matrix per expert.
static int pair_run_of_k(int N1, int K1, bool grouped1, int N2, int K2, bool grouped2) {
  const int nw = split_k_waves(N1, K1, grouped1), nw2 = split_k_waves(N2, K2, grouped2);
  if (nw2 <= nw) return K2;
  return ((K2 + 63) / 64 + nw2 / nw - 1) / (nw2 / nw) * 64;      // a multiple of 64: runs start at whole lines
}
TQ_API int tq_gemm_mfma_pair_splits(int N1, int K1, int grouped1, int N2, int K2, int grouped2) {
  const int k_per = pair_run_of_k(N1, K1, grouped1 != 0, N2, K2, grouped2 != 0);
  return (K2 + k_per - 1) / k_per;
}

TQ_API int tq_gemm_phases_pair_splits(int M1, int N1, int K1, int M2, int N2, int K2);

// Two products in one launch.  d1, d2: 20 numbers each, in the order of tq_gemm_mfma's arguments from `a`
// to `tile_rows`, then the gate's activation and the bits of the gated pair's limit as a float (0: none); both gated or
// both not, both into the same type.  Either
//  * few rows: both products that the streaming kernel takes 16 rows at a time (a matrix per expert with tile_rows 16, or
//    one matrix with M <= 16).  The waves that split k are those of the first product (the larger one by convention);
//  * or many, where tile_rows of the first is 64 + TQ_TILE_PAIRS (and a queue, as above): the first over experts by the row order's items, the second
//    of one matrix whose rows follow one another, k of either a multiple of 64 and 128 and more (gemm_phases.hip).
// splits2 > 1 (as tq_gemm_mfma_pair_splits says of few rows and tq_gemm_phases_pair_splits of many, for a plain second
// product into float): run z of its k goes to out + z * M * ldc, the bias to run 0.
TQ_API int tq_gemm_mfma_pair(const int64_t* d1, const int64_t* d2, int splits2, hipStream_t st) {
  MfmaGemmArgs g[2];
  int row_tiles[2];
  bool dual[2], out_act[2];
  const int64_t* d[2] = {d1, d2};
  int tile_rows1 = (int)d1[17];
  int* queue;
  if (!take_queue(tile_rows1, (const int*)d1[7], (const int*)d1[8], &queue)) return TQ_ERR_BAD_ARG;
  const bool many = tile_rows1 == 64 + TQ_TILE_PAIRS;
  for (int i = 0; i < 2; ++i) {
    const int64_t* p = d[i];
    const int M = (int)p[14], N = (int)p[15], K = (int)p[16], tile_rows = (int)p[17];
    if (M <= 0 || N <= 0 || K <= 0 || K % 8 != 0 || p[1] % 8 != 0 || p[6] % 8 != 0) return TQ_ERR_BAD_ARG;
    if (((uintptr_t)p[0] | (uintptr_t)p[4] | (uintptr_t)p[5]) % 16 != 0) return TQ_ERR_BAD_ARG;
    g[i] = MfmaGemmArgs{(const bf16_t*)p[0], p[1], (const int*)p[2], (int)p[3], (const bf16_t*)p[4], (const bf16_t*)p[5],
                        p[6], (const int*)p[7], (const int*)p[8], (const void*)p[9], (int)p[10], (void*)p[11], p[12],
                        M, N, K, K, 0, (int)p[18], 1, 0, 0.f};
    const uint32_t limit_bits = (uint32_t)p[19];
    memcpy(&g[i].limit, &limit_bits, sizeof(float));
    if (!(g[i].limit >= 0.f)) return TQ_ERR_BAD_ARG;
    if (g[i].gate < 0 || g[i].gate >= TQ_GATE_COUNT) return TQ_ERR_BAD_ARG;
    dual[i] = p[5] != 0;
    out_act[i] = p[13] != 0;
    if (many) {
      if (K % TBK || K < 2 * TBK || (i == 0 ? M % 64 || !g[i].tile_group : g[i].tile_group || g[i].a_rows)) return TQ_ERR_BAD_ARG;
      continue;
    }
    if (g[i].tile_group) {
      if (tile_rows != 16 || M % 16) return TQ_ERR_BAD_ARG;
      row_tiles[i] = M / 16;
    } else {
      if (M > 16) return TQ_ERR_BAD_ARG;
      row_tiles[i] = 1;
    }
  }
  if (dual[0] != dual[1] || out_act[0] != out_act[1]) return TQ_ERR_BAD_ARG;
  if (splits2 < 1) return TQ_ERR_BAD_ARG;
  if (many) {
    if (splits2 > 1) {
      if (dual[1] || out_act[1] || splits2 != tq_gemm_phases_pair_splits(g[0].M, g[0].N, g[0].K, g[1].M, g[1].N, g[1].K)) return TQ_ERR_BAD_ARG;
      g[1].k_per = (g[1].K / TBK + splits2 - 1) / splits2 * TBK;
      g[1].split_stride = (int64_t)g[1].M * g[1].ldc;
    }
    if (const int rc = launch_gemm_phases(g[0], &g[1], queue, dual[0], out_act[0], st)) return rc;
    TQ_LAUNCH_CHECK();
    return 0;
  }
  if (splits2 > 1) {
    if (dual[1] || out_act[1] || g[1].a_rows || g[1].tile_group) return TQ_ERR_BAD_ARG;
    g[1].k_per = pair_run_of_k(g[0].N, g[0].K, g[0].tile_group != nullptr, g[1].N, g[1].K, false);
    if (splits2 != (g[1].K + g[1].k_per - 1) / g[1].k_per) return TQ_ERR_BAD_ARG;
    g[1].split_stride = (int64_t)g[1].M * g[1].ldc;
  }
  const int nw = split_k_waves(g[0].N, g[0].K, g[0].tile_group != nullptr);
  const size_t shmem = nw > 1 ? (size_t)nw * (dual[0] ? 2 : 1) * 4 * 64 * sizeof(float) : 0;
  const int nx1 = (g[0].N + 15) / 16, nx2 = (g[1].N + 15) / 16;
  const int64_t n1 = (int64_t)nx1 * row_tiles[0], n2 = (int64_t)nx2 * row_tiles[1] * splits2;
  if (n1 + n2 > 0x7fffffff) return TQ_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)(n1 + n2));
  if (g[0].tile_group && !g[1].tile_group && lean_suits(g[0]) && lean_suits(g[1])) {
    const int cols = lean_columns(g[0], row_tiles[0], dual[0]), lx1 = g[0].N / cols, lx2 = g[1].N / cols, l2 = lx2 * splits2;
    if ((int64_t)lx1 * row_tiles[0] + l2 > 0x7fffffff) return TQ_ERR_UNSUPPORTED;
#define TQ_PAIR_OF(D, O, C) \
  hipLaunchKernelGGL((gemm_lean_pair_kernel<D, O, C>), dim3(lx1 * row_tiles[0] + l2), dim3(64 * nw), shmem, st, g[0], lx1, g[1], lx2, l2)
#define TQ_PAIR(D, O)                     \
  do {                                    \
    if (cols == 8) TQ_PAIR_OF(D, O, 8);   \
    else TQ_PAIR_OF(D, O, 16);            \
  } while (0)
    if (dual[0] && out_act[0]) TQ_PAIR(true, true);
    else if (dual[0]) TQ_PAIR(true, false);
    else if (out_act[0]) TQ_PAIR(false, true);
    else TQ_PAIR(false, false);
#undef TQ_PAIR
#undef TQ_PAIR_OF
    TQ_LAUNCH_CHECK();
    return 0;
  }
#define TQ_PAIR(D, O) \
  hipLaunchKernelGGL((gemm_stream_pair_kernel<D, O>), grid, dim3(64 * nw), shmem, st, g[0], nx1, g[1], nx2, row_tiles[1], (int)n2)
  if (dual[0] && out_act[0]) TQ_PAIR(true, true);
  else if (dual[0]) TQ_PAIR(true, false);
  else if (out_act[0]) TQ_PAIR(false, true);
  else TQ_PAIR(false, false);
#undef TQ_PAIR
  TQ_LAUNCH_CHECK();
  return 0;
}

// Queries, keys and values of T <= 16 tokens in one launch: a [T][K] bfloat16 (row stride lda) times w [(nh + 2 nkv)
// hd][K] plus bias, queries and keys rotated by positions[t] * inv_freq[d] on the pairs (d, d + hd / 2), queries to
// q_out [T][nh hd], keys and values into the pages (k_pool / v_pool with the layer's offset added; null: only the
// queries are made).  hd must be a multiple of 32 and the rotation span the whole head.
TQ_API int tq_qkv_rope_write(const void* a, int64_t lda, const void* w, const void* bias, int bias_type, int T, int K,
                             const int* positions, const int* seq_of_token, const int* block_table, int bt_stride,
                             const float* inv_freq, void* q_out, void* k_pool, void* v_pool, int page_size,
                             int64_t page_stride, int nh, int nkv, int hd, hipStream_t st) {
  if (T <= 0) return 0;
  if (T > 16 || hd % 32 != 0 || hd <= 0 || nh <= 0 || nkv <= 0) return TQ_ERR_UNSUPPORTED;
  if (K <= 0 || K % 8 != 0 || lda % 8 != 0 || ((uintptr_t)a | (uintptr_t)w) % 16 != 0) return TQ_ERR_BAD_ARG;
  if ((k_pool == nullptr) != (v_pool == nullptr) || page_size <= 0) return TQ_ERR_BAD_ARG;
  const int heads = k_pool ? nh + 2 * nkv : nh;
  const int N = (nh + 2 * nkv) * hd;
  MfmaGemmArgs g{(const bf16_t*)a, lda, nullptr, 1, (const bf16_t*)w, nullptr, 0, nullptr, nullptr, bias, bias_type,
                 nullptr, 0, T, N, K, K, 0, 0, 1};
  RopeWriteArgs p{positions, seq_of_token, block_table, bt_stride, inv_freq, (bf16_t*)q_out, (bf16_t*)k_pool,
                  (bf16_t*)v_pool, page_size, page_stride, nh, nkv, hd};
  int nw = split_k_waves(heads * hd / 2, K, false);
  if (nw > 8) nw = 8;
  const size_t shmem = (size_t)nw * 2 * 4 * 64 * sizeof(float);
  hipLaunchKernelGGL(qkv_rope_write_kernel, dim3(heads * (hd / 32)), dim3(64 * nw), shmem, st, g, p);
  TQ_LAUNCH_CHECK();
  return 0;
}
