// The gated delta rule of delta_rule.hip over long runs, in chunks of 32 tokens.  Which form a run takes is a matter of its own
// length alone (DC_FROM), so that what a sequence gets does not depend on the others of the step.
//
// With S the state before a chunk, G_t the decays of the chunk's tokens multiplied up to and with t (per key channel; one
// number for all of them in the form with a decay per head) and G_t / G_s the product of those behind s up to t:
//   u_t = beta_t (v_t - S^T (G_t k_t) - sum_{s < t} a_ts u_s),        a_ts = sum_d k_t[d] k_s[d] (G_t / G_s)[d]
//   o_t = S^T (G_t q_t) + sum_{s <= t} b_ts u_s,                       b_ts the same with q_t
//   S'  = G_32 S + sum_s (G_32 / G_s) k_s u_s^T
// so that u = U0 - W S with (I + beta a) [U0 | W] = beta [v | G k], a triangular system that does not hold the state.
// Two launches: delta_chunk_prep, every chunk and head side by side, works out U0, W, b and the decayed rows of q and k;
// delta_chunk_scan goes through a sequence's chunks in order with the state in registers.  Everything is float, on
// v_mfma_f32_16x16x4_f32 where it is a product.  No quotient is formed: a ratio G_t / G_s is the product of the factors
// between, and none is above one, whatever the decays.
//
// A step whose chunks do not fit the scratch (DC_SCRATCH) goes through it a window at a time: the same chunks of every run, so that
// the runs still go side by side, their state through memory from one window to the next; and so many runs at a time.
//
// Scratch (float), per chunk and head, in the order in which a wave's lanes of the scan take their operands (four floats a
// lane, 64 lanes a tile of 16 x 16): W [2 token tiles][D / 16] | G q alike | (G_32 / G) k [D / 16][2] | U0 [V / 16][2] |
// b [2][2] | G_32 [D].  Row 4 g + i of a tile of tokens is token 4 i + g: an instruction then takes four tokens that follow
// one another, and sums over tokens run in order, the latest and largest term last.
#include "delta_rule.h"

#define DC_T 32
// Tokens from which a run goes in chunks: a chunk costs the same whatever it holds, and the two launches 20 us before the first.
// Chunks and token by token, us, 16 heads of 128 x 128: one sequence of 32 tokens 24 and 23, of 48 25 and 30, of 96 27 and 51, of
// 1,024 90 and 475; 64 sequences of 32 tokens 195 and 212, of 48 295 and 288, of 64 302 and 364, of 256 970 and 1,291.  Heads of
// 256 x 256, whose scan kept 196 bytes a lane in scratch memory then: 38 and 42 for one of 48 tokens, 1,107 and 1,266 for 64 of them (without
// any, as now, both launches of 2,048 tokens of 8 heads of 256 x 128 take 222 us instead of 325).  Narrow heads in a
// crowded step, where a chunk's pairs weigh more than the state, are the exception: 64 sequences of 64 tokens and 32 heads of 64 x 64
// 225 and 215, 16 heads of 128 x 16 135 and 107, while one sequence of 256 tokens of these takes 27 and 127, 38 and 137.
#define DC_FROM 48
// Floats of scratch at the most (1 GiB), or those of one chunk: what a step of 30,000 tokens and 16 heads of 128 x 128 fills.  Beyond,
// a window's launches are a few more (us, in one window and in several of 1 GiB, 512 MiB and 256 MiB: 64 runs of 1,080 tokens 3,791,
// 3,980, 4,249 and 5,097; four of 32,768 7,007, 7,021, 7,137 and 7,346).
#define DC_SCRATCH (1 << 28)
typedef float dc_f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ __forceinline__ int64_t dc_floats(int D, int V) { return (int64_t)DC_T * (3 * D + V) + DC_T * DC_T + D; }

__device__ __forceinline__ int dc_chunks(int n) { return n >= DC_FROM ? (n + DC_T - 1) / DC_T : 0; }

// The chunks `first` to first + count - 1 of runs b0 to b0 + B - 1.
struct DeltaWindow {
  int b0, B, first, count;
};
// The token of row r of a tile, and the row of token r.
__device__ __forceinline__ int dc_turned(int r) { return 4 * (r % 4) + r / 4; }
// How many of its chunks a run of n tokens has there.
__device__ __forceinline__ int dc_inside(const DeltaWindow& w, int n) { return min(max(dc_chunks(n) - w.first, 0), w.count); }

// The run and the chunk of it that chunk number `want` of the window is, run by run; false behind the last one.  All 64 lanes of
// a wave call it together.
__device__ __forceinline__ bool dc_find(const int* __restrict__ cu_seqlens, const DeltaWindow& w, int want, int& b, int& c) {
  const int lane = threadIdx.x % TQ_WAVE;
  int base = 0;
  for (int b0 = w.b0; b0 < w.b0 + w.B; b0 += TQ_WAVE) {
    const int i = b0 + lane;
    const int own = i < w.b0 + w.B ? dc_inside(w, cu_seqlens[i + 1] - cu_seqlens[i]) : 0;
    int upto = own;
#pragma unroll
    for (int o = 1; o < TQ_WAVE; o *= 2) {
      const int before = __shfl_up(upto, o, TQ_WAVE);
      if (lane >= o) upto += before;
    }
    const uint64_t reached = __ballot(base + upto > want);
    if (reached) {
      const int at = __ffsll((unsigned long long)reached) - 1;
      b = b0 + at;
      c = w.first + want - base - (__shfl(upto, at, TQ_WAVE) - __shfl(own, at, TQ_WAVE));
      return true;
    }
    base += __shfl(upto, TQ_WAVE - 1, TQ_WAVE);
  }
  return false;
}

// grid (H, chunks of the window), block 512.  LDS: k, q, decays [32][LD] each, the products of the decays from the start of
// the token's half of the chunk up to and with it, and (in the decays' place) from behind it to the half's end (halves of 16:
// what lies between two tokens of different halves is one of each); the partial sums of a and b; a.
// The pairs of one half are formed channel by channel with the product of the decays between them (a lane keeps k_s times
// that product for D / 16 channels and walks through t); those of different halves are products of matrices, by waves 0 to 3
// while the others write the decayed rows out.  The waves' shares of a pair, and the products of decays, are put together in 64
// bits: a pair's rounding stands alone where token by token the state's rows round each by itself, and would weigh more.
// The triangular system then takes a column of its right side to a thread.
// A workgroup is a chain of such steps with a barrier between (19 us alone); two of 80 KB share a compute unit, and 2,048 tokens of
// 16 heads of 128 x 128, 1,024 workgroups, take 59 us (79 with loads under conditions, each of which is waited for at once).
template <int ND, bool HEAD>
__global__ __launch_bounds__(512, 4) void delta_chunk_prep_kernel(const float* __restrict__ qn, const float* __restrict__ kn,
                                                               const float* __restrict__ vc, const float* __restrict__ beta,
                                                               const float* __restrict__ ag, const float* __restrict__ a_log,
                                                               const float* __restrict__ dt_bias,
                                                               const int* __restrict__ cu_seqlens, DeltaWindow window, DeltaDims dm,
                                                               float* __restrict__ scratch) {
  constexpr int D = 16 * ND, LD = D + 4, SHARES = 8 * 512 > DC_T * LD ? 8 * 512 : DC_T * LD;
  extern __shared__ __align__(16) float dc_lds[];
  float* ks = dc_lds;
  float* qs = ks + DC_T * LD;
  float* gs = qs + DC_T * LD;
  float* down = gs;                      // products from behind t to the half's end, once the pairs are formed
  float* up = gs + DC_T * LD;            // products from the half's start up to t; before that
  float* part = up;                      // [wave][a, b][16][16], the waves' shares of the pairs of one half
  float* across = up + SHARES;           // [wave][a, b][16][16], the waves' shares of the pairs across
  float* am = across + 4 * 512;          // [32][36] beta_t a_ts
  float* bt = am + DC_T * 36;            // [32]
  const int h = blockIdx.x, tid = threadIdx.x, wave = tid / TQ_WAVE, lane = tid % TQ_WAVE;
  const int H = dm.H, G = dm.G, V = dm.V, gq = h / (H / G);
  int b, c;
  if (!dc_find(cu_seqlens, window, blockIdx.y, b, c)) return;
  b = __builtin_amdgcn_readfirstlane(b);      // (alike in every lane, and so are the addresses made from them)
  c = __builtin_amdgcn_readfirstlane(c);
  const int t0 = cu_seqlens[b] + c * DC_T, nc = min(DC_T, cu_seqlens[b + 1] - t0);
  float* w_out = scratch + ((size_t)blockIdx.y * H + h) * dc_floats(D, V);
  float* q_out = w_out + DC_T * D;
  float* k_out = q_out + DC_T * D;
  float* u_out = k_out + DC_T * D;
  float* b_out = u_out + DC_T * V;
  float* g_out = b_out + DC_T * DC_T;

  // rows behind the run's end: q = k = beta = 0, decay 1
  const float rate = HEAD ? 0.f : expf(a_log[h]);
  // (every load is unconditional, of the run's last token where there is none: a load under a condition is waited for at once)
#pragma unroll 2
  for (int idx = tid; idx < DC_T * D / 4; idx += 512) {
    const int t = idx / (D / 4), d = 4 * (idx % (D / 4)), tc = t0 + min(t, nc - 1);
    const size_t row = (size_t)tc * G * D + (size_t)gq * D + d;
    dc_f32x4 k = *reinterpret_cast<const dc_f32x4*>(kn + row);
    dc_f32x4 q = *reinterpret_cast<const dc_f32x4*>(qn + row);
    dc_f32x4 g;
    if (HEAD) {
      const float one = ag[(size_t)tc * H + h];
      g = dc_f32x4{one, one, one, one};
    } else {
      g = *reinterpret_cast<const dc_f32x4*>(ag + (size_t)tc * (H * D + H * V) + (size_t)h * D + d);
#pragma unroll
      for (int i = 0; i < 4; ++i) g[i] = expf(-rate * softplus_f(g[i] + dt_bias[h * D + d + i]));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      k[i] = t < nc ? k[i] : 0.f;
      q[i] = t < nc ? q[i] : 0.f;
      g[i] = t < nc ? g[i] : 1.f;
    }
    *reinterpret_cast<dc_f32x4*>(ks + t * LD + d) = k;
    *reinterpret_cast<dc_f32x4*>(qs + t * LD + d) = q;
    *reinterpret_cast<dc_f32x4*>(gs + t * LD + d) = g;
  }
  if (tid < DC_T) bt[tid] = tid < nc ? beta[(size_t)(t0 + tid) * H + h] : 0.f;
  __syncthreads();
  // pairs of one half: wave w takes half w % 2 and a quarter of the channels, a lane token s and a sixteenth of the channels
  {
    const int first = wave % 2 * 16, s = lane % 16, d0 = (wave / 2 * 4 + lane / 16) * ND;
    float kp[ND];
    unsigned own[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      own[i] = __float_as_uint(ks[(first + s) * LD + d0 + i]);
      kp[i] = 0.f;
    }
    float* to = part + wave * 512;
#pragma unroll 1
    for (int t4 = 0; t4 < 16; t4 += 4) {
      float a[4], bb[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t4 + j;
        const float* kt = ks + (first + t) * LD + d0;
        const float* qt = qs + (first + t) * LD + d0;
        const float* gt = gs + (first + t) * LD + d0;
        const unsigned starts = t == s ? 0xffffffffu : 0u;      // (kp is zero until then)
        a[j] = bb[j] = 0.f;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
          kp[i] = fmaf(kp[i], gt[i], __uint_as_float(own[i] & starts));
          a[j] = fmaf(kt[i], kp[i], a[j]);
          bb[j] = fmaf(qt[i], kp[i], bb[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = with_lane_xor<16>(a[j], LanesSum());
        bb[j] = with_lane_xor<16>(bb[j], LanesSum());
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = with_lane_xor<32>(a[j], LanesSum());
        bb[j] = with_lane_xor<32>(bb[j], LanesSum());
      }
      if (lane < 16)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          to[(t4 + j) * 16 + s] = a[j];
          to[256 + (t4 + j) * 16 + s] = bb[j];
        }
    }
  }
  __syncthreads();
  const int pt = tid / 16 % 16, ps = tid % 16;              // the pair of a 16 x 16 block that this thread puts together
  const int b_at = (dc_turned(pt) + 16 * (ps % 4)) * 4 + ps / 4;      // and its place in b's tiles
  {
    const int half = tid / 256, i = tid % 256;
    double a = 0., bb = 0.;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      a += part[(half + 2 * w) * 512 + i];
      bb += part[(half + 2 * w) * 512 + 256 + i];
    }
    am[(16 * half + pt) * 36 + 16 * half + ps] = ps < pt ? (float)(bt[16 * half + pt] * a) : 0.f;
    b_out[3 * half * 256 + b_at] = ps <= pt ? (float)bb : 0.f;
  }
  __syncthreads();
  for (int idx = tid; idx < 2 * D; idx += 512) {
    const int first = idx / D * 16, d = idx % D;
    float g[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) g[i] = gs[(first + i) * LD + d];
    double p = 1.;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      p *= g[i];
      up[(first + i) * LD + d] = (float)p;
    }
    p = 1.;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      down[(first + i) * LD + d] = (float)p;
      p *= g[i];
    }
  }
  __syncthreads();
  if (wave < 4) {
    // pairs across: rows 16 .. 31 by columns 0 .. 15, a quarter of the channels to a wave
    const int r = lane % 16, g4 = lane / 16;
    dc_f32x4 ca = {0.f, 0.f, 0.f, 0.f}, cb = ca;
    for (int db = wave; db < ND; db += 4) {
      const int d = 16 * db + 4 * g4;
      const dc_f32x4 kt = *reinterpret_cast<const dc_f32x4*>(ks + (16 + r) * LD + d);
      const dc_f32x4 qt = *reinterpret_cast<const dc_f32x4*>(qs + (16 + r) * LD + d);
      const dc_f32x4 pt4 = *reinterpret_cast<const dc_f32x4*>(up + (16 + r) * LD + d);
      const dc_f32x4 kc = *reinterpret_cast<const dc_f32x4*>(ks + r * LD + d);
      const dc_f32x4 pc = *reinterpret_cast<const dc_f32x4*>(down + r * LD + d);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float col = kc[i] * pc[i];
        ca = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[i] * pt4[i], col, ca, 0, 0, 0);
        cb = __builtin_amdgcn_mfma_f32_16x16x4f32(qt[i] * pt4[i], col, cb, 0, 0, 0);
      }
    }
    float* sum = across + wave * 512;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sum[(4 * g4 + i) * 16 + r] = ca[i];
      sum[256 + (4 * g4 + i) * 16 + r] = cb[i];
    }
  } else {
    // q and k with their decays, in the scan's order
    const int tid2 = tid - 256;
    for (int idx = tid2; idx < 2 * ND * 64; idx += 256) {
      const int l = idx % 64, tile = idx / 64, tb = tile / ND, db = tile % ND;
      const int t = 16 * tb + dc_turned(l % 16), d = 16 * db + 4 * (l / 16);
      const dc_f32x4 q = *reinterpret_cast<const dc_f32x4*>(qs + t * LD + d);
      dc_f32x4 p = *reinterpret_cast<const dc_f32x4*>(up + t * LD + d);
      if (tb) p *= *reinterpret_cast<const dc_f32x4*>(up + 15 * LD + d);
      *reinterpret_cast<dc_f32x4*>(q_out + (size_t)idx * 4) = q * p;
    }
    for (int idx = tid2; idx < ND * 2 * 64; idx += 256) {
      const int l = idx % 64, tile = idx / 64, db = tile / 2, tb = tile % 2;
      const int d = 16 * db + l % 16, t = 16 * tb + l / 16;
      const float rest = tb ? 1.f : up[31 * LD + d];
      dc_f32x4 k;
#pragma unroll
      for (int i = 0; i < 4; ++i) k[i] = ks[(t + 4 * i) * LD + d] * down[(t + 4 * i) * LD + d] * rest;
      *reinterpret_cast<dc_f32x4*>(k_out + (size_t)idx * 4) = k;
    }
    for (int d = tid2; d < D; d += 256) g_out[d] = up[15 * LD + d] * up[31 * LD + d];
  }
  __syncthreads();
  if (tid < 256) {
    double a = 0., bb = 0.;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      a += across[w * 512 + tid];
      bb += across[w * 512 + 256 + tid];
    }
    am[(16 + pt) * 36 + ps] = (float)(bt[16 + pt] * a);
    b_out[2 * 256 + b_at] = (float)bb;
  }
  __syncthreads();
  // the triangular system, a column to a thread
  for (int col = tid; col < V + D; col += 512) {
    const bool is_v = col < V;
    float x[DC_T];
    if (is_v) {
      const float* from = vc + (size_t)t0 * H * V + (size_t)h * V;
#pragma unroll
      for (int t = 0; t < DC_T; ++t) x[t] = (from + (size_t)min(t, nc - 1) * H * V)[col];
#pragma unroll
      for (int t = 0; t < DC_T; ++t) x[t] = t < nc ? bt[t] * x[t] : 0.f;
    } else {
      const int d = col - V;
      const float first_half = up[15 * LD + d];
#pragma unroll
      for (int t = 0; t < DC_T; ++t) x[t] = bt[t] * (ks[t * LD + d] * (up[t * LD + d] * (t < 16 ? 1.f : first_half)));
    }
    // (the fences keep the compiler from asking for all rows of a at once)
#pragma unroll
    for (int t = 1; t < DC_T; ++t) {
      asm volatile("" ::: "memory");
      dc_f32x4 a[DC_T / 4];
#pragma unroll
      for (int s4 = 0; s4 < (t + 3) / 4; ++s4) a[s4] = *reinterpret_cast<const dc_f32x4*>(am + t * 36 + 4 * s4);
      // (the sum by itself, then off x: its terms are smaller than x, and so are the roundings on the way)
      float y = 0.f, z = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) {
        if (s % 2) z = fmaf(a[s / 4][s % 4], x[s], z);
        else y = fmaf(a[s / 4][s % 4], x[s], y);
      }
      x[t] -= y + z;
    }
    if (is_v) {
#pragma unroll
      for (int f = 0; f < DC_T / 4; ++f)      // tile (col / 16, f / 4), lane col % 16 + 16 (f % 4)
        *reinterpret_cast<dc_f32x4*>(u_out + ((size_t)(col / 16 * 2 + f / 4) * 64 + col % 16 + 16 * (f % 4)) * 4) =
            dc_f32x4{x[f / 4 * 16 + f % 4], x[f / 4 * 16 + f % 4 + 4], x[f / 4 * 16 + f % 4 + 8], x[f / 4 * 16 + f % 4 + 12]};
    } else {
#pragma unroll
      for (int t = 0; t < DC_T; ++t)           // tile (t / 16, d / 16), lane of t's row + 16 (d % 16 / 4), number d % 4 of channel d
        w_out[((size_t)(t / 16 * ND + (col - V) / 16) * 64 + dc_turned(t % 16) + 16 * ((col - V) % 16 / 4)) * 4 + (col - V) % 4] = -x[t];
    }
  }
}

// grid (H V / 16, runs of the window), block 256: a workgroup takes 16 value channels of a head through the sequence's chunks in the window;
// wave w keeps the rows of the state in key tiles w, w + 4, ... as accumulators, which are the operands of the products with the state as
// they stand (the key channels of a product are taken in the order 0, 4, 8, 12, 1, 5, ...).  Each wave's share of u passes
// through LDS, one barrier a chunk; its share of o, to which waves 0, 1 and 2 add one of b's three tiles each once u is known,
// goes along with the next chunk's u.  In the loop the next two chunks' operands are on their way meanwhile.  The blocks of a head lie H apart, so
// that they run on one die (H a multiple of 8) and share what they read in its L2.
// A chunk is a chain: 8 NB products with the state, the exchange, in whose time 8 NB more are formed for o, and 8 NB into the state, 1.5 us of
// which 0.64 are the products'.  2,048 tokens of 16 heads of 128 x 128, us: 97; 119 before with a wait for all loads on their way every two
// chunks (see the loop; 116 without), the products for o in front of the exchange (109 behind it) and the key tiles' chains one behind the
// other under conditions of their own.  Level: b's products between those into the state.  (Token by token both launches' work took 0.94 ms, 0.45
// us a token.)
// WHOLE: every wave has NB key tiles (D = 64 NB), so that nothing is under a condition and the tiles' chains of products go on side by side.
template <int NB, bool WHOLE>
__global__ __launch_bounds__(256, NB < 4 ? 2 : 1) void delta_chunk_scan_kernel(const float* __restrict__ scratch,
                                                               const int* __restrict__ cu_seqlens,
                                                               const int* __restrict__ slots, float* __restrict__ state,
                                                               int64_t state_stride, DeltaWindow window, DeltaDims dm,
                                                               float* __restrict__ o_raw) {
  __shared__ __align__(16) float ex[2][4][4][256];      // [buffer][wave][u, u, the chunk before's o, o][lane][4]
  const int H = dm.H, D = WHOLE ? 64 * NB : dm.D, V = dm.V, ND = D / 16, VB = V / 16;
  const int h = blockIdx.x % H, vb = blockIdx.x / H, b = window.b0 + blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TQ_WAVE), lane = threadIdx.x % TQ_WAVE, r = lane % 16, g4 = lane / 16;
  int t0 = cu_seqlens[b], n = cu_seqlens[b + 1] - t0;
  const int chunks = dc_inside(window, n);
  if (chunks == 0) return;
  int base = 0;
  for (int i = window.b0 + lane; i < b; i += TQ_WAVE) base += dc_inside(window, cu_seqlens[i + 1] - cu_seqlens[i]);
#pragma unroll
  for (int o = TQ_WAVE / 2; o > 0; o >>= 1) base += __shfl_xor(base, o, TQ_WAVE);
  base = __builtin_amdgcn_readfirstlane(base);
  t0 += window.first * DC_T;      // (chunks count from the window's first on)
  n -= window.first * DC_T;
  const size_t chunk_floats = dc_floats(D, V);
  const float* at = scratch + ((size_t)base * H + h) * chunk_floats;
  float* S = state + (size_t)slots[b] * state_stride + (size_t)h * D * V + vb * 16 + r;
  dc_f32x4 s[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int db = wave + 4 * j;
#pragma unroll
    for (int i = 0; i < 4; ++i) s[j][i] = WHOLE || db < ND ? S[(size_t)(16 * db + 4 * g4 + i) * V] : 0.f;
  }
  const dc_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  struct Operands {
    dc_f32x4 w[2][NB], q[2][NB], k[NB][2], g[NB], u0[2], bq;
  };
  // (tiles that a wave does not have are fetched from its first one and take no part)
  auto fetch = [&](Operands& to, int chunk) {
    const float* c = at + (size_t)chunk * H * chunk_floats;
    auto tile = [&](int i) { return reinterpret_cast<const dc_f32x4*>(c + (size_t)i * 256)[lane]; };
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int db = WHOLE || wave + 4 * j < ND ? wave + 4 * j : 0;
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        to.w[tb][j] = tile(tb * ND + db);
        to.q[tb][j] = tile(2 * ND + tb * ND + db);
        to.k[j][tb] = tile(4 * ND + db * 2 + tb);
      }
      to.g[j] = reinterpret_cast<const dc_f32x4*>(c + (size_t)DC_T * (3 * D + V) + DC_T * DC_T + 16 * db)[g4];
    }
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) to.u0[tb] = tile(6 * ND + vb * 2 + tb);
    to.bq = tile(6 * ND + 2 * VB + (wave == 0 ? 0 : wave == 1 ? 2 : 3));      // b's tile (0, 0), (1, 0) or (1, 1)
  };
  dc_f32x4 po[2] = {zero, zero};      // this wave's share of the o of the chunk that has its u
  // two numbers of the o of chunk c from the waves' shares, in wave order: token tile wave / 2, rows 4 g4 + 2 (wave % 2) and the next
  auto read_out = [&](const float (*from)[4][256], int c, bool last) {
    float y0 = 0.f, y1 = 0.f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      const float2 y = *reinterpret_cast<const float2*>(&from[ww][2 + wave / 2][lane * 4 + 2 * (wave % 2)]);
      y0 += y.x, y1 += y.y;
    }
    const int t = 16 * (wave / 2) + 8 * (wave % 2) + g4;
    float* row = o_raw + ((size_t)(t0 + c * DC_T) * H + h) * V + vb * 16 + ((size_t)t * H * V + r);
    if (!last || c * DC_T + t < n) row[0] = y0;
    if (!last || c * DC_T + t + 4 < n) row[(size_t)4 * H * V] = y1;
  };
  // (neither loads nor stores are under a condition, or the compiler would wait for all loads on their way at each use of some)
  auto one_chunk = [&](int c, Operands& in, bool first) {
    dc_f32x4 pu[2], next[2];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      pu[tb] = zero;
      next[tb] = zero;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (WHOLE || wave + 4 * j < ND)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) pu[tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(in.w[tb][j][i], s[j][i], pu[tb], 0, 0, 0);
    }
    float (*to)[4][256] = ex[c & 1];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      *reinterpret_cast<dc_f32x4*>(&to[wave][tb][lane * 4]) = pu[tb];
      *reinterpret_cast<dc_f32x4*>(&to[wave][2 + tb][lane * 4]) = po[tb];
    }
    __syncthreads();
    // the waves' shares in wave order, and U0; they come out of LDS while the products for o are formed
    dc_f32x4 u[2], share[2][4];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) share[tb][ww] = *reinterpret_cast<const dc_f32x4*>(&to[ww][tb][lane * 4]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (WHOLE || wave + 4 * j < ND)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) next[tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(in.q[tb][j][i], s[j][i], next[tb], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      u[tb] = share[tb][0];
#pragma unroll
      for (int ww = 1; ww < 4; ++ww) u[tb] += share[tb][ww];
      u[tb] += in.u0[tb];
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) s[j] *= in.g[j];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (WHOLE || wave + 4 * j < ND) s[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(in.k[j][tb][i], u[tb][i], s[j], 0, 0, 0);
    if (!first) read_out(to, c - 1, false);
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) po[tb] = next[tb];
    if (wave < 3) {
      const dc_f32x4 us = wave == 2 ? u[1] : u[0];
      dc_f32x4 y = wave == 0 ? next[0] : next[1];
      const dc_f32x4 before = y;
#pragma unroll
      for (int i = 0; i < 4; ++i) y = __builtin_amdgcn_mfma_f32_16x16x4f32(in.bq[i], us[i], y, 0, 0, 0);
      // A value that is not finite in a later token of the tile meets the zeros of b: the earlier tokens' sums are formed
      // again without it.
      bool strange = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) strange |= !(fabsf(y[i]) <= 3.402823466e38f);
      if (wave != 1 && __any(strange)) {
        y = before;
#pragma unroll 1
        for (int t = 0; t < 16; ++t) {
          const float mine_u = t / 4 == 0 ? us[0] : t / 4 == 1 ? us[1] : t / 4 == 2 ? us[2] : us[3];
          const float mine_b = t / 4 == 0 ? in.bq[0] : t / 4 == 1 ? in.bq[1] : t / 4 == 2 ? in.bq[2] : in.bq[3];
          const float ut = __shfl(mine_u, r + 16 * (t % 4), TQ_WAVE);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float bt = __shfl(mine_b, 4 * g4 + i + 16 * (t % 4), TQ_WAVE);
            if (t <= 4 * i + g4) y[i] = fmaf(bt, ut, y[i]);
          }
        }
      }
      if (wave == 0) po[0] = y;
      else po[1] = y;
    }
    fetch(in, min(c + 2, chunks - 1));
  };
  // Pairs behind the first chunk or the first two, so that the loop holds nothing but whole pairs: with a single chunk behind them the
  // compiler made one body of both, and waited at its head for all loads on their way to move what they bring to other registers.
  // Those first chunks ask for their operands as they begin, and the loop asks again for what the last of them asked for.  Tried instead: the first
  // two on their way together, and the loop beginning with what is on its way already; the body is longer then, and slower (both launches, us with
  // one body, so tried and as it is: 64 tokens of 16 heads of 128 x 128 26.1, 25.6 and 25.0, 128 29.6, 28.6 and 28.2, 256 36.8, 34.8 and 34.1, 2,048
  // 164, 147 and 144, 3,001 236, 210 and 206; 64 tokens of 8 of 256 x 128 38.3, 35.5 and 34.6).
  Operands even, odd;
  fetch(even, 0);
  one_chunk(0, even, true);
  int c = 1;
  if (chunks % 2 == 0) {
    fetch(odd, 1);
    one_chunk(1, odd, false);
    c = 2;
  }
  if (c < chunks) {
    fetch(even, c);
    fetch(odd, c + 1);
#pragma unroll 1
    for (; c < chunks; c += 2) {
      one_chunk(c, even, false);
      one_chunk(c + 1, odd, false);
    }
  }
  float (*to)[4][256] = ex[chunks & 1];
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) *reinterpret_cast<dc_f32x4*>(&to[wave][2 + tb][lane * 4]) = po[tb];
  __syncthreads();
  read_out(to, chunks - 1, true);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int db = wave + 4 * j;
    if (WHOLE || db < ND)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[(size_t)(16 * db + 4 * g4 + i) * V] = s[j][i];
  }
}

// The most chunks that the long runs of T tokens of B sequences have: each begins one beyond its whole ones.
static int64_t dc_bound(int T, int B) { return (int64_t)T / DC_T + (B < T / DC_FROM ? B : T / DC_FROM); }

// Sizes that the tiles take.
static bool dc_takes(int D, int V) { return D % 16 == 0 && D <= 256 && V % 16 == 0 && V > 0; }

// Chunks that the scratch holds.
static int64_t dc_held(int H, int D, int V) {
  const int64_t n = DC_SCRATCH / (H * dc_floats(D, V));
  return n < 1 ? 1 : n < 65535 ? n : 65535;
}

// Floats of scratch that tq_delta_chunks needs for T tokens of B sequences; 0 where no run can be long enough for chunks, or the
// sizes do not fit the tiles.
TQ_API int64_t tq_delta_chunk_scratch(int T, int B, int H, int D, int V) {
  if (!dc_takes(D, V) || H < 1 || B < 1 || B > 65535 || T < DC_FROM) return 0;
  const int64_t all = dc_bound(T, B), held = dc_held(H, D, V);
  return (all < held ? all : held) * H * dc_floats(D, V);
}

// What tq_delta_scan (head_decay 0; ag is only read) and tq_delta_scan_h (head_decay 1; ag [T][H] decays, a_log and dt_bias
// null) compute, over `scratch`: runs of DC_FROM tokens and more in chunks, the others token by token in a launch of their own.
// longest, shortest: bounds that the host knows for the runs' tokens (T and 0 if it knows none).
TQ_API int tq_delta_chunks(const float* qn, const float* kn, const float* vc, const float* beta, const float* ag,
                           const float* a_log, const float* dt_bias, int head_decay, const int* cu_seqlens, const int* slots,
                           float* state, int64_t state_stride, int H, int G, int D, int V, int taps, int T, int B,
                           int longest, int shortest, float* scratch, float* o_raw, hipStream_t st) {
  if (B <= 0 || T <= 0) return 0;
  const DeltaDims d{H, G, D, V, taps, head_decay ? 0 : 1, head_decay ? 0 : 1, head_decay ? 1 : 0};
  if (H < 1 || G < 1 || H % G || taps < 1 || taps > 64 || state_stride < dd_state(d) || !scratch || !ag || (!head_decay && (!a_log || !dt_bias)))
    return TQ_ERR_BAD_ARG;
  if (!dc_takes(D, V) || B > 65535 || T < DC_FROM) return TQ_ERR_UNSUPPORTED;
  if (longest < 0 || longest > T) return TQ_ERR_BAD_ARG;
  const int nd = D / 16;
  const int row = DC_T * (D + 4);
  const size_t shmem = (size_t)(3 * row + (row > 8 * 512 ? row : 8 * 512) + 4 * 512 + DC_T * 36 + DC_T) * sizeof(float);
  auto launch = [&](const DeltaWindow& w, unsigned chunks) -> int {
#define TQ_PREP(N, HD)                                                                                                       \
  do {                                                                                                                       \
    if (shmem > 48 * 1024 && hipFuncSetAttribute((const void*)delta_chunk_prep_kernel<N, HD>,                               \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)      \
      return TQ_ERR_UNSUPPORTED;                                                                                             \
    hipLaunchKernelGGL((delta_chunk_prep_kernel<N, HD>), dim3(H, chunks), dim3(512), shmem, st, qn, kn, vc, beta, ag, a_log, \
                       dt_bias, cu_seqlens, w, d, scratch);                                                                  \
  } while (0)
#define TQ_PREP_CASE(N)               \
  case N:                             \
    if (head_decay) TQ_PREP(N, true); \
    else TQ_PREP(N, false);           \
    break;
    switch (nd) {
      TQ_PREP_CASE(1) TQ_PREP_CASE(2) TQ_PREP_CASE(3) TQ_PREP_CASE(4) TQ_PREP_CASE(5) TQ_PREP_CASE(6) TQ_PREP_CASE(7)
      TQ_PREP_CASE(8) TQ_PREP_CASE(9) TQ_PREP_CASE(10) TQ_PREP_CASE(11) TQ_PREP_CASE(12) TQ_PREP_CASE(13) TQ_PREP_CASE(14)
      TQ_PREP_CASE(15) TQ_PREP_CASE(16)
    }
#undef TQ_PREP_CASE
#undef TQ_PREP
    const dim3 grid((unsigned)(H * (V / 16)), w.B);
#define TQ_SCAN(NB)                                                                                                                \
  hipLaunchKernelGGL((nd == 4 * NB ? delta_chunk_scan_kernel<NB, true> : delta_chunk_scan_kernel<NB, false>), grid, dim3(256), 0, st, scratch, cu_seqlens, slots, state, state_stride, w, d, o_raw)
    if (nd <= 4) TQ_SCAN(1);
    else if (nd <= 8) TQ_SCAN(2);
    else TQ_SCAN(4);
#undef TQ_SCAN
    TQ_LAUNCH_CHECK();
    return 0;
  };
  // windows of as many chunks of every run as the scratch surely holds
  const int held = (int)dc_held(H, D, V), last = longest / DC_T + (longest % DC_T ? 1 : 0);
  for (int b0 = 0; b0 < B; b0 += held) {
    DeltaWindow w{b0, B - b0 < held ? B - b0 : held, 0, 0};
    const int64_t all = dc_bound(T, w.B);
    for (; w.first < last; w.first += w.count) {
      // runs that go on behind the windows before: each has more tokens than those took, and the DC_FROM that make it long
      const int64_t tokens = (int64_t)w.first * DC_T + 1, most = T / (tokens > DC_FROM ? tokens : DC_FROM), runs = w.B < most ? w.B : most;
      if (runs == 0) break;
      const int64_t count = all <= held ? last : held / runs;
      w.count = (int)(count < last - w.first ? count : last - w.first);
      if (int rc = launch(w, (unsigned)(all < runs * w.count ? all : runs * w.count))) return rc;
    }
  }
  if (shortest >= DC_FROM) return 0;
  return delta_short_runs(qn, kn, vc, beta, ag, a_log, dt_bias, cu_seqlens, slots, state, state_stride, d, DC_FROM, T, B, o_raw, st);
}
