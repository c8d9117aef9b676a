// Routing of tokens to experts: router logits, softmax, top-k, and the order of (token, expert)
// pairs by expert that the expert products work through.
#include "common.h"

// ---------------------------------------------------------------- router
// Two kernels.  router_logits: logit[t][e] = sum_j x[t][j] * wr[e][j] in float
// (/root/reference/src/engine/tq_moe.c:611-618), with the shared expert's gate vector as one more row.  A
// wave takes one row of wr (or a few) at a time for a group of up to 8 tokens whose activations wait in LDS; lane l sums
// a fixed share of the elements and the lanes' sums are added by a butterfly: one order for every token,
// whatever else is in the batch.  Rows are dealt over a second grid dimension when
// there are few tokens, so that decoding does not leave the chip to eight waves.
// What bounds it: loads in a chain (a workgroup's activations, then its rows of wr), and for many tokens the multiply-adds and the sums
// over the lanes.  So a workgroup asks for all its tokens' activations before it stores the first, and a wave's 32 sums change places on
// the way (62 exchanges instead of 192 shuffles and additions).  us with the choice, before and now, 60 experts of 2,048 and a shared one,
// bf16: one token 7.3 and 6.6, 97 8.8 and 7.8, 512 14.6 and 10.5, 1,733 27.7 and 17.6, 2,048 24.4 and 16.9, 11,000 93.7 and 66.1;
// 256 experts, 2,048 tokens 76.2 and 53.3; 32-bit, 16,385 tokens 140 and 103.
// router_select, one wave per token: top-k by logit, k rounds of a search in which >= lets the highest index
// win among equal logits, so ids come out by descending logit (tq_moe.c:626-645).  Weights:
//   renorm != 0: softmax over the selected logits (tq_moe.c:648-678), times wscale;
//   renorm == 0: softmax over all experts, the selected probabilities kept as they are;
//   renorm == TQ_ROUTE_SIGMOID: every expert's score is the sigmoid of its logit, the choice is by score, and the weights
//     are the selected scores over (their sum + 1e-20), times wscale.  With TQ_ROUTE_PAIR_GROUPS added, a group's score is
//     the sum of its two largest scores.
// shared_gate[t] = 1 / (1 + exp(-(x . shared_w)))  (tq_moe.c:1012-1018, with an exact exponential).
#define TQ_ROUTE_SIGMOID 2
#define TQ_ROUTE_PAIR_GROUPS 4
#define RT 8   // most tokens per workgroup of router_logits
#define TQ_ROUTER_MANY 240   // tokens from which on a workgroup of router_logits has eight waves and RT tokens
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load4(const float* p, float* w) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p);
  w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
}
__device__ __forceinline__ void load4(const bf16_t* p, float* w) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  w[0] = __uint_as_float(v.x << 16);
  w[1] = __uint_as_float(v.x & 0xffff0000u);
  w[2] = __uint_as_float(v.y << 16);
  w[3] = __uint_as_float(v.y & 0xffff0000u);
}

// The sums over the wave of N values (a power of two up to the wave's lanes): afterwards s[0] of lanes i * 64 / N and on is value i's.
// Each value's is the sum that wave_sum gives, in its order, by fewer steps: at a step two values change places by halves, and one
// addition makes the next sums of both.
template <int N, int O>
__device__ __forceinline__ void wave_sums(float* s) {
  if constexpr (N > 1) {
    const bool upper = (threadIdx.x & O) != 0;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const float a = s[i], b = s[i + N / 2];
      if constexpr (O >= 16) {
        typedef unsigned two __attribute__((ext_vector_type(2)));
        const two t = __builtin_bit_cast(two, O == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                                                      : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false));
        s[i] = __uint_as_float(t.x) + __uint_as_float(t.y);
      } else {
        const float own = upper ? b : a;
        s[i] = with_lane_xor<O>(upper ? a : b, [own](float, float other) { return own + other; });
      }
    }
    wave_sums<N / 2, O / 2>(s);
  } else if constexpr (O > 0) {
    s[0] = with_lane_xor<O>(s[0], LanesSum());
    wave_sums<1, O / 2>(s);
  }
}

// TG: tokens per workgroup (tokens beyond T are zeros in LDS and are not stored).  RW: rows of wr that a wave
// takes at a time, so that one read of the activations from LDS serves RW rows.  Neither changes the order in
// which a logit is summed: of every 512 elements lane l sums 4 l .. 4 l + 3 and 256 + 4 l .. 256 + 4 l + 3 (its
// 16-byte reads from LDS then lie side by side with its neighbours'), block after block.  In LDS a token's row is
// filled with zeros up to a multiple of 512, so the last block needs no predicate: there the weights are read
// from the row's last elements instead, and multiplied by zeros.
// xs: [TG][Hp] of LDS.  The workgroup takes the rows of its part out of `parts`; logit (token k of its, row e) goes to out[k * rows + e].
template <class W, int TG, int RW, int TH>
__device__ __forceinline__ void token_logits(const float* __restrict__ x, const W* __restrict__ wr, const W* __restrict__ shared_w, int rows,
                                             int E, float* out, int T, int H, const float* __restrict__ bias, float* xs, int part, int parts) {
  const int Hp = (H + 511) / 512 * 512;
  const int t0 = blockIdx.x * TG;
  const int nt = min(TG, T - t0);
  const int wave = threadIdx.x / TQ_WAVE, lane = threadIdx.x % TQ_WAVE;
  const bool vec = H % 4 == 0;
  if (vec) {
    const int Hp4 = Hp / 4, H4 = H / 4;
    f32x4* dst = reinterpret_cast<f32x4*>(xs);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int j = threadIdx.x; j < Hp4; j += TH) {
      f32x4 v[TG];
#pragma unroll
      for (int k = 0; k < TG; ++k) v[k] = k < nt && j < H4 ? reinterpret_cast<const f32x4*>(x + (size_t)(t0 + k) * H)[j] : zero;
#pragma unroll
      for (int k = 0; k < TG; ++k) dst[k * Hp4 + j] = v[k];
    }
  } else {
    for (int i = threadIdx.x; i < TG * Hp; i += TH) {
      const int k = i / Hp, j = i % Hp;
      xs[i] = k < nt && j < H ? x[(size_t)(t0 + k) * H + j] : 0.f;
    }
  }
  __syncthreads();
  // workgroups start at different rows, so that they do not all ask for the same row at once
  const int rot = (blockIdx.x * 5) % rows;
  for (int idx = (part * (TH / TQ_WAVE) + wave) * RW; idx < rows; idx += parts * (TH / TQ_WAVE) * RW) {
    const W* row[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int i = min(idx + r, rows - 1) + rot;
      const int e = i < rows ? i : i - rows;
      row[r] = e < E ? wr + (size_t)e * H : shared_w;
    }
    float s[RW * TG];
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int k = 0; k < TG; ++k) s[r * TG + k] = 0.f;
    if (vec) {
      const f32x4* xv = reinterpret_cast<const f32x4*>(xs);
      const int Hp4 = Hp / 4;
      constexpr int NB = RW >= 4 ? 2 : 4;      // blocks whose weights are asked for before the first is used
      for (int b0 = 0; b0 < Hp; b0 += NB * 512) {
        float w[NB][RW][8];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
          const int b = b0 + u * 512;
          const int g0 = min(b + 4 * lane, H - 4), g1 = min(b + 256 + 4 * lane, H - 4);
#pragma unroll
          for (int r = 0; r < RW; ++r) {
            load4(row[r] + g0, &w[u][r][0]);
            load4(row[r] + g1, &w[u][r][4]);
          }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
          const int b = b0 + u * 512;
          if (b < Hp) {
#pragma unroll
            for (int k = 0; k < TG; ++k) {
              const f32x4 a = xv[k * Hp4 + b / 4 + lane];
              const f32x4 c = xv[k * Hp4 + b / 4 + 64 + lane];
#pragma unroll
              for (int r = 0; r < RW; ++r) {
                float v = s[r * TG + k];
                v = fmaf(a.x, w[u][r][0], v);
                v = fmaf(a.y, w[u][r][1], v);
                v = fmaf(a.z, w[u][r][2], v);
                v = fmaf(a.w, w[u][r][3], v);
                v = fmaf(c.x, w[u][r][4], v);
                v = fmaf(c.y, w[u][r][5], v);
                v = fmaf(c.z, w[u][r][6], v);
                v = fmaf(c.w, w[u][r][7], v);
                s[r * TG + k] = v;
              }
            }
          }
        }
      }
    } else {
      for (int j = lane; j < H; j += TQ_WAVE) {
#pragma unroll
        for (int r = 0; r < RW; ++r) {
          const float w = to_f32(row[r][j]);
#pragma unroll
          for (int k = 0; k < TG; ++k) s[r * TG + k] = fmaf(xs[k * Hp + j], w, s[r * TG + k]);
        }
      }
    }
    wave_sums<RW * TG, TQ_WAVE / 2>(s);
    constexpr int LANES = TQ_WAVE / (RW * TG);      // that hold one sum
    const int r = lane / LANES / TG, k = lane / LANES % TG;
    if (lane % LANES == 0 && k < nt && idx + r < rows) {      // (a bias per expert, not for the shared expert's gate row)
      const int i = idx + r + rot, at = i < rows ? i : i - rows;
      out[(size_t)k * rows + at] = bias && at < E ? s[0] + bias[at] : s[0];
    }
  }
}

template <class W, int TG, int RW, int TH>
__global__ __launch_bounds__(TH, TH == 512 ? 4 : 1) void router_logits_kernel(const float* __restrict__ x, const W* __restrict__ wr,
                                                            const W* __restrict__ shared_w, int rows, int E,
                                                            float* __restrict__ logits, int T, int H,
                                                            const float* __restrict__ bias) {
  extern __shared__ __attribute__((aligned(16))) float xs[];      // [TG][Hp]
  token_logits<W, TG, RW, TH>(x, wr, shared_w, rows, E, logits + (size_t)blockIdx.x * TG * rows, T, H, bias, xs, blockIdx.y, gridDim.y);
}

// The group score of every lane's group where groups are runs of PER neighbouring lanes (a power of two): its largest value or, with
// `two`, the sum of its two largest.
template <int PER, int O = PER / 2>
__device__ __forceinline__ void best_two(float& m, float& m2) {
  if constexpr (O > 0) {
    const float om = __shfl_xor(m, O, TQ_WAVE), om2 = __shfl_xor(m2, O, TQ_WAVE);
    m2 = fmaxf(fminf(m, om), fmaxf(m2, om2));
    m = fmaxf(m, om);
    best_two<PER, O / 2>(m, m2);
  }
}

// As select_token below where a lane holds NL experts (lane and lane + 64) and no logit is NaN, with the same results: nothing goes
// through LDS, and a round of the search is a maximum over the wave in the vector unit and a ballot (the highest of the experts that hold
// it) instead of twelve shuffles.  One token's choice and order 4.4 us instead of 7.4, eight tokens' 5.6 (8.2), the choice of
// 2,048 tokens 5.0 (13.5), 60 experts, four per token.  Lane k returns the k-th expert chosen; the caller stores it.
template <int NL>
__device__ __forceinline__ int select_small(const float (&logit)[NL], int E, int topk, int renorm, int groups, int keep,
                                            float* __restrict__ weights, float* __restrict__ shared_gate, const float (&corr)[NL],
                                            bool corrected, int n_real, float wscale) {
  const int lane = threadIdx.x % TQ_WAVE;
  const bool sigmoid = (renorm & TQ_ROUTE_SIGMOID) != 0, pair_groups = (renorm & TQ_ROUTE_PAIR_GROUPS) != 0;
  bool mine[NL];
  float v[NL];
#pragma unroll
  for (int u = 0; u < NL; ++u) {
    mine[u] = lane + u * TQ_WAVE < E;
    v[u] = mine[u] ? logit[u] : -INFINITY;
  }
  auto largest = [&]() {
    float m = v[0];
#pragma unroll
    for (int u = 1; u < NL; ++u) m = fmaxf(m, v[u]);
    return wave_max(m);
  };
  float mx = 0.f, denom = 1.f;
  if (!renorm) {
    mx = largest();
    float d = 0.f;
#pragma unroll
    for (int u = 0; u < NL; ++u)
      if (mine[u]) d += expf(v[u] - mx);
    denom = wave_sum(d);
  }
#pragma unroll
  for (int u = 0; u < NL; ++u) {
    if (sigmoid && mine[u]) v[u] = 1.0f / (1.0f + expf(-v[u]));
    if (corrected && mine[u]) v[u] = expf(v[u] - mx) * (1.0f / denom) + corr[u];
  }
  if constexpr (NL == 1) {
    if (groups > 1 && keep < groups) {
      const int per = E / groups;
      float m = v[0], m2 = -INFINITY;
      switch (per) {
        case 2: best_two<2>(m, m2); break;
        case 4: best_two<4>(m, m2); break;
        case 8: best_two<8>(m, m2); break;
        case 16: best_two<16>(m, m2); break;
        case 32: best_two<32>(m, m2); break;
      }
      if (pair_groups && per > 1) m += m2;
      const int group = lane / per;
      int better = 0;
      for (int g2 = 0; g2 < groups; ++g2) {
        const float other = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(m), g2 * per));
        better += (other > m || (other == m && g2 > group)) ? 1 : 0;
      }
      if (better >= keep) v[0] = -INFINITY;
    }
  }
  float sel = 0.f;
  int sel_id = -1;
  for (int k = 0; k < topk; ++k) {
    const float best = largest();
    int bi = 0;      // (none: only if every score is NaN, through its correction)
    float raw = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(logit[0])));
#pragma unroll
    for (int u = 0; u < NL; ++u) {      // (the later, the higher the index)
      const unsigned long long at = __ballot(mine[u] && v[u] == best);
      if (at) {
        const int l = 63 - __builtin_clzll(at);
        bi = u * TQ_WAVE + l;
        raw = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(logit[u]), l));
      }
    }
    if (lane == k) {
      sel = corrected ? raw : best;
      sel_id = bi;
    }
#pragma unroll
    for (int u = 0; u < NL; ++u)
      if (lane + u * TQ_WAVE == bi) v[u] = -INFINITY;
  }
  if (sigmoid) {
    const float s = wave_sum(lane < topk ? sel : 0.f);
    if (lane < topk) weights[lane] = sel / (s + 1e-20f) * wscale;
  } else if (renorm) {
    const float m = wave_max(lane < topk ? sel : -INFINITY);
    const float p = lane < topk ? expf(sel - m) : 0.f;
    const float s = wave_sum(p);
    if (lane < topk) weights[lane] = (s > 0.f ? p * (1.0f / s) : 0.f) * wscale;
  } else {
    const float wgt = lane < topk ? expf(sel - mx) * (1.0f / denom) : 0.f;
    if (lane < topk) weights[lane] = wgt;
    if (n_real < E) {
      const float idw = wave_sum(sel_id >= n_real ? wgt : 0.f);
      if (lane == 0) shared_gate[0] = idw;
    }
  }
  return sel_id;
}
// A token's choice by select_small where it takes it: up to 64 experts, in groups of powers of two or none, or up to 128 without
// groups, and no logit that is NaN.  Lane k receives the k-th expert.
template <int NL>
__device__ __forceinline__ bool chosen_small(const float* __restrict__ src, int rows, int E, int topk, int renorm, int groups, int keep,
                                             float* __restrict__ weights, float* __restrict__ shared_gate,
                                             const float* __restrict__ correction, int n_real, float wscale, int& e) {
  const int lane = threadIdx.x % TQ_WAVE;
  float logit[NL], corr[NL];
  bool nan = false;
#pragma unroll
  for (int u = 0; u < NL; ++u) {
    const int at = min(lane + u * TQ_WAVE, E - 1);
    logit[u] = src[at];
    corr[u] = correction ? correction[at] : 0.f;
  }
  const float own = rows > E ? src[E] : 0.f;
#pragma unroll
  for (int u = 0; u < NL; ++u) nan = nan || logit[u] != logit[u];
  if (__any(nan)) return false;
  if (rows > E && lane == 0) shared_gate[0] = 1.0f / (1.0f + expf(-own));
  e = select_small<NL>(logit, E, topk, renorm, groups, keep, weights, shared_gate, corr, correction != nullptr, n_real, wscale);
  return true;
}
__device__ __forceinline__ bool choose_small(const float* __restrict__ src, int rows, int E, int topk, int renorm, int groups, int keep,
                                             float* __restrict__ weights, float* __restrict__ shared_gate,
                                             const float* __restrict__ correction, int n_real, float wscale, int& e) {
  const bool grouped = groups > 1 && keep < groups;
  if (E <= TQ_WAVE && !(grouped && ((E / groups) & (E / groups - 1))))
    return chosen_small<1>(src, rows, E, topk, renorm, groups, keep, weights, shared_gate, correction, n_real, wscale, e);
  if (E <= 2 * TQ_WAVE && !grouped)
    return chosen_small<2>(src, rows, E, topk, renorm, groups, keep, weights, shared_gate, correction, n_real, wscale, e);
  return false;
}

// One wave chooses for one token.  src: the token's `rows` logits; lg: E floats of LDS for this wave; ids,
// weights, shared_gate: where the token's results go; ids2: a second place for the ids (LDS), or null.
// groups > 1: the experts form `groups` equal groups of neighbours; a group's score is its largest logit (the order of
// softmax scores is the order of logits), only experts of the `keep` best groups can be chosen (among groups of
// equal score the highest index wins, as among experts), and the softmax over all experts is taken before the
// others are left out.
__device__ __forceinline__ void select_token(const float* __restrict__ src, int rows, int E, int topk, int renorm,
                                             int groups, int keep, float* lg, int* __restrict__ ids, int* ids2,
                                             float* __restrict__ weights, float* __restrict__ shared_gate,
                                             const float* __restrict__ correction = nullptr, int n_real = 1 << 30,
                                             float wscale = 1.0f) {
  const int lane = threadIdx.x % TQ_WAVE;
  const bool sigmoid = (renorm & TQ_ROUTE_SIGMOID) != 0, pair_groups = (renorm & TQ_ROUTE_PAIR_GROUPS) != 0;
  if (int e; choose_small(src, rows, E, topk, renorm, groups, keep, weights, shared_gate, correction, n_real, wscale, e)) {
    if (lane < topk) {
      ids[lane] = e;
      if (ids2) ids2[lane] = e;
    }
    return;
  }
  for (int e = lane; e < E; e += TQ_WAVE) lg[e] = src[e];
  if (rows > E && lane == 0) shared_gate[0] = 1.0f / (1.0f + expf(-src[E]));
  __builtin_amdgcn_wave_barrier();
  float mx = 0.f, denom = 1.f;
  if (!renorm) {      // softmax over all experts, before any logit is taken out
    mx = -INFINITY;
    for (int e = lane; e < E; e += TQ_WAVE) mx = fmaxf(mx, lg[e]);
    mx = wave_max(mx);
    float d = 0.f;
    for (int e = lane; e < E; e += TQ_WAVE) d += expf(lg[e] - mx);
    denom = wave_sum(d);
  }
  if (sigmoid) {
    for (int e = lane; e < E; e += TQ_WAVE) lg[e] = 1.0f / (1.0f + expf(-lg[e]));
    __builtin_amdgcn_wave_barrier();
  }
  if (correction) {
    // the choice is by the softmax score plus a number per expert; the weights are the scores without it
    for (int e = lane; e < E; e += TQ_WAVE) lg[e] = expf(lg[e] - mx) * (1.0f / denom) + correction[e];
    __builtin_amdgcn_wave_barrier();
  }
  if (groups > 1 && keep < groups) {
    const int per = E / groups;
    // a lane per group (in turns of 64): the group's largest logit, or the sum of its two largest scores
    float gmax[4];      // up to 256 groups
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int gi = lane + 64 * i;
      float m = -INFINITY, m2 = -INFINITY;
      if (gi < groups)
        for (int e = gi * per; e < (gi + 1) * per; ++e) {
          m2 = fmaxf(m2, fminf(m, lg[e]));      // the second largest so far
          m = fmaxf(m, lg[e]);
        }
      gmax[i] = pair_groups && per > 1 ? m + m2 : m;
    }
    // a group is kept if fewer than `keep` groups are better: a larger best logit, or the same and a higher index (the
    // order in which rounds of a search would take them, without the rounds: every lane looks at every group once)
    unsigned kept = 0;      // bit i: group lane + 64 i is kept
    int better[4] = {0, 0, 0, 0};
    for (int g2 = 0; g2 < groups; ++g2) {
      const int src = g2 % 64;
      float other = __shfl(gmax[0], src, TQ_WAVE);
      if (groups > 64) {
        const float o1 = __shfl(gmax[1], src, TQ_WAVE), o2 = __shfl(gmax[2], src, TQ_WAVE), o3 = __shfl(gmax[3], src, TQ_WAVE);
        other = g2 < 64 ? other : g2 < 128 ? o1 : g2 < 192 ? o2 : o3;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int gi = lane + 64 * i;
        better[i] += (other > gmax[i] || (other == gmax[i] && g2 > gi)) ? 1 : 0;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (lane + 64 * i < groups && better[i] < keep) kept |= 1u << i;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int gi = lane + 64 * i;
      if (gi < groups && !((kept >> i) & 1u))
        for (int e = gi * per; e < (gi + 1) * per; ++e) lg[e] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
  }
  float sel = 0.f;    // lane k keeps the k-th selected logit
  int sel_id = -1;    // and its expert
  for (int k = 0; k < topk; ++k) {
    float bv = -INFINITY;
    int bi = -1;
    for (int e = lane; e < E; e += TQ_WAVE) {
      const float v = lg[e];
      if (v >= bv) {     // e ascends: the highest index among equals
        bv = v;
        bi = e;
      }
    }
#pragma unroll
    for (int o = TQ_WAVE / 2; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, TQ_WAVE);
      const int oi = __shfl_xor(bi, o, TQ_WAVE);
      if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) {
        bv = ov;
        bi = oi;
      }
    }
    if (bi < 0) bi = 0;   // only if every logit is NaN
    if (lane == k) {
      sel = correction ? src[bi] : bv;
      sel_id = bi;
    }
    if (lane == 0) {
      ids[k] = bi;
      if (ids2) ids2[k] = bi;
      lg[bi] = -INFINITY;   // taken out of the later rounds
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (sigmoid) {
    const float s = wave_sum(lane < topk ? sel : 0.f);
    if (lane < topk) weights[lane] = sel / (s + 1e-20f) * wscale;
  } else if (renorm) {
    const float m = wave_max(lane < topk ? sel : -INFINITY);
    const float p = lane < topk ? expf(sel - m) : 0.f;
    const float s = wave_sum(p);
    if (lane < topk) weights[lane] = (s > 0.f ? p * (1.0f / s) : 0.f) * wscale;
  } else {
    const float wgt = lane < topk ? expf(sel - mx) * (1.0f / denom) : 0.f;
    if (lane < topk) weights[lane] = wgt;
    if (n_real < E) {     // experts from n_real on are the identity: the sum of their weights multiplies the token's own row
      const float idw = wave_sum(sel_id >= n_real ? wgt : 0.f);
      if (lane == 0) shared_gate[0] = idw;
    }
  }
}

__global__ __launch_bounds__(256) void router_select_kernel(const float* __restrict__ logits, int rows, int E,
                                                            int topk, int renorm, int groups, int keep,
                                                            int* __restrict__ ids, float* __restrict__ weights,
                                                            float* __restrict__ shared_gate, int T,
                                                            const float* __restrict__ correction, int n_real,
                                                            float wscale) {
  extern __shared__ float sm[];      // [4][E]
  const int wave = threadIdx.x / TQ_WAVE;
  const int t = blockIdx.x * 4 + wave;
  if (t >= T) return;
  select_token(logits + (size_t)t * rows, rows, E, topk, renorm, groups, keep, sm + wave * E, ids + (size_t)t * topk, nullptr,
               weights + (size_t)t * topk, shared_gate + t, correction, n_real, wscale);
}

static int launch_router_logits(const float* x, const void* wr, const void* shared_w, int wtype, int E,
                                float* logits, int T, int H, hipStream_t st, const float* bias = nullptr) {
  const int rows = E + (shared_w ? 1 : 0);
  const size_t hp = ((size_t)H + 511) / 512 * 512;      // a token's row in LDS
  // Many tokens: 8 of them to a workgroup of eight waves, whatever LDS they take (a wave's read of 4 rows of wr serves 8 tokens).  The
  // other form and this one, with the choice, us, 60 experts of 2,048 and a shared one: 160 tokens 8.4 and 8.6, 333 10.7 and 10.1,
  // 512 12.9 and 10.5, 700 15.9 and 11.8; 256 experts: 64 16.5 and 16.5, 240 22.2 and 19.5, 512 27.3 and 24.2; rows of 3,584, 114 KB
  // of LDS, 2,048 tokens 42.7 and 33.1.
  const bool many = T >= TQ_ROUTER_MANY && hp * RT * sizeof(float) <= 160 * 1024;
  // Where two such workgroups do not share a unit (rows beyond 2,560), two of 4 tokens that do take as long for the same 8 tokens, 1.10 times as
  // long with 256 experts and 0.85 with 16; but a last round of up to half the units then takes half a round, and a whole one with 8 (us with 8
  // and with 4 tokens, the choice among them; rows of 3,584: 256 experts, 2,049 tokens 132 and 112, 3,072 136 and 121, 3,073 136 and 145, 4,096 142 and
  // 156, 4,097 205 and 187, 8,192 273 and 296, 10,300 350 and 340, 13,197 458 and 469; 128 experts, 3,001 73 and 63, 4,096 78 and 81, 13,197 246 and
  // 243; 64, 2,049 39 and 33, 4,096 47 and 47, 13,197 145 and 133; 16, 8,192 46 and 40; rows of 3,072, 4,096 and 5,120 alike).
  const bool wide = many && T > 2048 && hp * RT * sizeof(float) > 80 * 1024 &&
                    (E <= 64 || ((T - 1) % 2048 < 1024 && T <= (E <= 128 ? 16384 : 12288)));
  int tg = wide ? 4 : RT;
  while (!many && tg > 1 && (size_t)tg * hp * sizeof(float) > 32 * 1024) tg /= 2;   // small enough for several workgroups per CU
  const size_t shmem = (size_t)tg * hp * sizeof(float);
  if (shmem > 160 * 1024) return TQ_ERR_UNSUPPORTED;
  const int groups = (T + tg - 1) / tg, waves = many ? 8 : 4;
  // The rows are dealt over so many workgroups that the chip holds about 2048 of them: what a wave does is a
  // chain of loads, and only many waves hide it.  A wave takes 1, 2 or 4 rows at a time.
  int row_groups = (many ? 512 : 2048) / groups;
  row_groups = row_groups < 1 ? 1 : (row_groups > (rows + waves - 1) / waves ? (rows + waves - 1) / waves : row_groups);
  const int rows_per_wave = (rows + row_groups * waves - 1) / (row_groups * waves);
  const int rw = rows_per_wave >= 4 ? 4 : (rows_per_wave >= 2 ? 2 : 1);
#define TQ_ROUTER(TGV, RWV, THV)                                                                                    \
  do {                                                                                                              \
    if (shmem > 48 * 1024)                                                                                          \
      (void)hipFuncSetAttribute((const void*)router_logits_kernel<W, TGV, RWV, THV>,                                \
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);                                  \
    hipLaunchKernelGGL((router_logits_kernel<W, TGV, RWV, THV>), dim3(groups, row_groups), dim3(THV), shmem, st, x, \
                       (const W*)wr, (const W*)shared_w, rows, E, logits, T, H, bias);                              \
  } while (0)
#define TQ_ROUTER_RW(TGV, THV)              \
  do {                                      \
    if (rw == 4) TQ_ROUTER(TGV, 4, THV);    \
    else if (rw == 2) TQ_ROUTER(TGV, 2, THV); \
    else TQ_ROUTER(TGV, 1, THV);            \
  } while (0)
  TQ_DISPATCH_W(wtype, {
    if (wide) TQ_ROUTER_RW(4, 512);
    else if (many) TQ_ROUTER_RW(8, 512);
    else if (tg == 8) TQ_ROUTER_RW(8, 256);
    else if (tg == 4) TQ_ROUTER_RW(4, 256);
    else if (tg == 2) TQ_ROUTER_RW(2, 256);
    else TQ_ROUTER_RW(1, 256);
  });
#undef TQ_ROUTER_RW
#undef TQ_ROUTER
  TQ_LAUNCH_CHECK();
  return 0;
}

// logits: scratch of T * (E + 1) floats (T * E without a shared gate vector).
// Whether a choice within the best `keep` of `groups` groups of experts can be made: groups == 1 means none.
static int groups_ok(int E, int topk, int groups, int keep) {
  if (groups == 1) return 1;
  return groups >= 1 && groups <= 256 && E % groups == 0 && keep >= 1 && keep <= groups && topk <= keep * (E / groups);
}

// bias (null, or float [E]): added to the experts' logits before the choice.
static int router_topk_impl(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E,
                            int topk, int renorm, int groups, int keep, int* ids, float* weights, float* shared_gate,
                            float* logits, int T, int H, hipStream_t st, const float* correction, int n_real, float wscale = 1.0f) {
  if (T <= 0) return 0;
  if (topk < 1 || topk > 64 || topk > E || E > 8192) return TQ_ERR_UNSUPPORTED;
  if (!groups_ok(E, topk, groups, keep)) return TQ_ERR_BAD_ARG;
  const int rc = launch_router_logits(x, wr, shared_w, wtype, E, logits, T, H, st, bias);
  if (rc) return rc;
  const int rows = E + (shared_w ? 1 : 0);
  hipLaunchKernelGGL(router_select_kernel, dim3((T + 3) / 4), dim3(256), (size_t)4 * E * sizeof(float), st, logits,
                     rows, E, topk, renorm, groups, keep, ids, weights, shared_gate, T, correction, n_real, wscale);
  TQ_LAUNCH_CHECK();
  return 0;
}

TQ_API int tq_router_topk_biased(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E,
                                 int topk, int renorm, int groups, int keep, int* ids, float* weights, float* shared_gate,
                                 float* logits, int T, int H, hipStream_t st) {
  return router_topk_impl(x, wr, shared_w, bias, wtype, E, topk, renorm, groups, keep, ids, weights, shared_gate, logits, T, H,
                          st, nullptr, E);
}

TQ_API int tq_router_topk_grouped(const float* x, const void* wr, const void* shared_w, int wtype, int E, int topk,
                                  int renorm, int groups, int keep, int* ids, float* weights, float* shared_gate,
                                  float* logits, int T, int H, hipStream_t st) {
  return tq_router_topk_biased(x, wr, shared_w, nullptr, wtype, E, topk, renorm, groups, keep, ids, weights, shared_gate,
                               logits, T, H, st);
}

TQ_API int tq_router_topk(const float* x, const void* wr, const void* shared_w, int wtype, int E, int topk,
                          int renorm, int* ids, float* weights, float* shared_gate, float* logits, int T, int H,
                          hipStream_t st) {
  return tq_router_topk_grouped(x, wr, shared_w, wtype, E, topk, renorm, 1, 1, ids, weights, shared_gate, logits, T, H, st);
}

// ---------------------------------------------------------------- order of pairs by expert
// Pair i = (token i / topk, its (i % topk)-th expert ids[i]).  Pairs are put in order of expert and,
// within an expert, of i (a stable counting sort, so the order never depends on timing).  Each
// expert's run of rows starts at a multiple of `unit` rows so that a row tile of the expert
// products belongs to one expert; the rows between are marked -1.
//   sorted_token[r]  token whose activations feed row r, or -1
//   pair_slot[i]     row of pair i
//   tile_expert[j]   expert of row tile j (tiles of `unit` rows), n_tiles[0] tiles in all
//   tile_expert[cap / unit + p]   first row tile of item p, n_tiles[1] items in all: an expert's row tiles two or, where
//                    TQ_ITEMS_OF_FOUR is added to `unit`, four at a time (its last item holds what is left), for the product
//                    that takes several tiles of one expert per workgroup; item p ends where item p + 1 begins, the last one
//                    at n_tiles[0]
// One workgroup of 16 waves does all of it.  Wave w owns the w-th sixteenth of the pairs: it goes through
// them 64 at a time, finds for every lane the lanes that hold the same expert (a ballot per bit of the expert's
// number), gives it its rank among them in order of lane and adds their number to its count of the expert.
// After a barrier the counts of all waves give every expert's first row and every wave's first row within
// the expert, and each pair's row is that plus its rank.
#define AW 16   // waves (one where a single token is ordered: the result does not depend on their number)

// One wave goes through its pairs seg_beg .. seg_end - 1, 64 at a time: every lane finds the lanes that hold the same
// expert (a ballot per bit of the expert's number), takes its rank among the wave's pairs of that expert so far, in
// order of pair, and the expert's first lane adds the batch's number to the wave's count mine[e].  The rank goes to
// pair_slot[i], or, with one_batch (at most 64 pairs a wave), stays with the lane in my_e, my_rank.
__device__ __forceinline__ void rank_segment(const int* ids, int seg_beg, int seg_end, int E, int* mine,
                                             int* __restrict__ pair_slot, bool one_batch, int& my_e, int& my_rank) {
  const int lane = threadIdx.x % TQ_WAVE;
  for (int b = seg_beg; b < seg_end; b += TQ_WAVE) {
    const int i = b + lane;
    const bool valid = i < seg_end;
    const int e = valid ? ids[i] : -1;
    // the lanes that hold the same expert: one ballot per bit of the expert's number
    unsigned long long same = __ballot(valid);
    for (int bit = 0; (1 << bit) < E; ++bit) {
      const unsigned long long set = __ballot(valid && ((e >> bit) & 1));
      same &= ((e >> bit) & 1) ? set : ~set;
    }
    const unsigned long long lower = same & ((1ull << lane) - 1ull);
    const int base = mine[valid ? e : 0];
    const int rank = base + __popcll(lower);
    __builtin_amdgcn_wave_barrier();       // every lane has read its count before the expert's first lane adds to it
    if (valid && lower == 0) mine[e] = base + __popcll(same);
    __builtin_amdgcn_wave_barrier();
    if (one_batch) {
      my_e = e;
      my_rank = rank;
    } else if (valid) {
      pair_slot[i] = rank;      // rank within (wave, expert) for now
    }
  }
}

// A wave zeroes the queues behind n_tiles (16..47; n_tiles[2] is the number of experts with rows then), if there are any, and takes what
// says so off the row tiles of an item; false: there are none.
#define TQ_WITH_QUEUES 256
__device__ __forceinline__ bool clear_queues(int* __restrict__ n_tiles, int& per_item) {
  if (!(per_item & TQ_WITH_QUEUES)) return false;
  per_item -= TQ_WITH_QUEUES;
  if (threadIdx.x % TQ_WAVE < 32) n_tiles[16 + threadIdx.x % TQ_WAVE] = 0;
  return true;
}

// Wave 0 of a workgroup turns the experts' padded sizes starts[e] into their first rows (an exclusive scan, each lane
// a contiguous run of experts) and (`write`) writes the row tiles' experts, the items and their numbers.
__device__ __forceinline__ void scan_starts(int* starts, int E, int unit, int per_item, int cap,
                                            int* __restrict__ tile_expert, int* __restrict__ n_tiles, bool write = true) {
  const int lane = threadIdx.x % TQ_WAVE;
  const bool queues = write && clear_queues(n_tiles, per_item);
  {
    const int chunk = (E + TQ_WAVE - 1) / TQ_WAVE;
    const int e0 = lane * chunk, e1 = min(E, e0 + chunk);
    int sum = 0, isum = 0, live = 0;
    for (int e = e0; e < e1; ++e) {
      sum += starts[e];
      live += starts[e] > 0;
      isum += (starts[e] / unit + per_item - 1) / per_item;
    }
    const int incl = wave_scan_add(sum), iincl = wave_scan_add(isum);
    int row = incl - sum, item = iincl - isum;
    int* items = tile_expert + cap / unit;
    for (int e = e0; e < e1; ++e) {
      const int padded = starts[e];
      starts[e] = row;
      for (int j = 0; write && j < padded / unit; ++j) {
        tile_expert[row / unit + j] = e;
        if (j % per_item == 0) items[item++] = row / unit + j;
      }
      row += padded;
    }
    const int used = queues ? wave_scan_add(live) : 0;
    if (write && lane == TQ_WAVE - 1) {
      n_tiles[0] = incl / unit;
      n_tiles[1] = iincl;
      if (queues) n_tiles[2] = used;
    }
  }
}

// ids may lie in LDS or in memory; cnt: (NW + 1) * E ints of LDS ([NW][E] counts, then E starts).  All NW waves
// of the workgroup call it together.
template <int NW>
__device__ __forceinline__ void align_pairs(const int* ids, int n_pairs, int E, int topk, int unit, int per_item, int cap,
                                            int* __restrict__ sorted_token, int* __restrict__ pair_slot,
                                            int* __restrict__ tile_expert, int* __restrict__ n_tiles, int* cnt,
                                            int n_real = 1 << 30) {
  // (experts from n_real on have no matrices: their pairs get no rows, pair_slot -1, and they no tiles)
  int* starts = cnt + NW * E;
  const int wave = threadIdx.x / TQ_WAVE, lane = threadIdx.x % TQ_WAVE;
  for (int i = threadIdx.x; i < cap; i += blockDim.x) sorted_token[i] = -1;
  for (int i = threadIdx.x; i < NW * E; i += blockDim.x) cnt[i] = 0;
  __syncthreads();
  const int per = ((n_pairs + NW - 1) / NW + TQ_WAVE - 1) / TQ_WAVE * TQ_WAVE;   // pairs per wave, whole batches
  const int seg_beg = wave * per, seg_end = min(n_pairs, seg_beg + per);
  int* mine = cnt + wave * E;
  // with at most 64 pairs per wave a thread meets its pair again in the last loop (i == threadIdx.x both times):
  // expert and rank stay in its registers and need not go through memory
  const bool one_batch = per == TQ_WAVE;
  int my_e = -1, my_rank = 0;
  rank_segment(ids, seg_beg, seg_end, E, mine, pair_slot, one_batch, my_e, my_rank);
  __syncthreads();
  // counts become each wave's first row within its expert; starts[e] first holds the expert's padded size
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int total = 0;
    for (int w = 0; w < NW; ++w) {
      const int c = cnt[w * E + e];
      cnt[w * E + e] = total;
      total += c;
    }
    starts[e] = e < n_real ? (total + unit - 1) / unit * unit : 0;
  }
  __syncthreads();
  if (wave == 0) scan_starts(starts, E, unit, per_item, cap, tile_expert, n_tiles);
  __syncthreads();
  if (one_batch) {
    if (my_e >= n_real) {
      pair_slot[threadIdx.x] = -1;
    } else if (my_e >= 0) {
      const int i = threadIdx.x;
      const int r = starts[my_e] + cnt[wave * E + my_e] + my_rank;
      pair_slot[i] = r;
      sorted_token[r] = i / topk;
    }
    return;
  }
  for (int i = threadIdx.x; i < n_pairs; i += blockDim.x) {
    const int e = ids[i], w = i / per;
    if (e >= n_real) {
      pair_slot[i] = -1;
      continue;
    }
    const int r = starts[e] + cnt[w * E + e] + pair_slot[i];
    pair_slot[i] = r;
    sorted_token[r] = i / topk;
  }
}

__global__ __launch_bounds__(64 * AW) void moe_align_kernel(const int* __restrict__ ids, int n_pairs, int E,
                                                            int topk, int unit, int per_item, int cap,
                                                            int* __restrict__ sorted_token,
                                                            int* __restrict__ pair_slot,
                                                            int* __restrict__ tile_expert,
                                                            int* __restrict__ n_tiles, int n_real) {
  extern __shared__ int cnt[];
  align_pairs<AW>(ids, n_pairs, E, topk, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, cnt, n_real);
}

// The choice and the same order by many workgroups, for steps of more than a handful of tokens: two launches.
//  * route_choose: a workgroup of eight waves has the logits of its TG tokens in LDS, a wave each chooses for them, and one wave ranks their
//    pairs and leaves how many each expert has in table[workgroup][e];
//  * route_place: every workgroup adds the table up for itself, all of it for the experts' first rows (the first workgroup writes the row tiles
//    and items from them) and what stands before its own segments (a segment: the pairs of one workgroup of route_choose), and gives its pairs their rows.
// The results are those of the one workgroup: pairs in order of expert and, within an expert, of pair.
// What bounds them is waiting: a launch, the activations, the rows of wr twice, the choice; and a launch, the table, two barriers, a pair's
// rank.  us by logits, choice and order apart (five launches; six from 8,192 pairs on) and by these, in a graph: 60 experts of 2,048 and a
// shared one, four a token: 513 tokens 19.0 and 16.1, 1,024 20.6 and 17.4, 2,048 26.8 and 22.3, 3,001 38.3 and 29.5, 8,192 62.5 and 55.2; 32
// of 1,024: 2,048 tokens 19.7 and 13.7; 64 of 3,584, eight a token: 1,500 48.3 and 31.6, 4,096 69.2 and 60.9; 256 experts, 2,048 tokens 78.2
// and 63.3.
template <class W, int TG>
__global__ __launch_bounds__(512, 4) void route_choose_kernel(const float* __restrict__ x, const W* __restrict__ wr, const W* __restrict__ shared_w,
                                                              int rows, int E, int T, int H, const float* __restrict__ bias, int topk, int renorm,
                                                              int groups, int keep, const float* __restrict__ correction, int n_real,
                                                              float wscale, int* __restrict__ ids, float* __restrict__ weights,
                                                              float* __restrict__ shared_gate, int cap, int* __restrict__ sorted_token,
                                                              int* __restrict__ pair_slot, int* __restrict__ table) {
  extern __shared__ __attribute__((aligned(16))) float xs[];      // [TG][Hp], then [TG][rows] logits, [TG][E] of the choice, [TG][topk] ids, [E] counts
  const int Hp = (H + 511) / 512 * 512, t0 = blockIdx.x * TG, nt = min(TG, T - t0), wave = threadIdx.x / TQ_WAVE;
  float* logits = xs + TG * Hp;
  float* lg = logits + TG * rows;
  int* ids_l = (int*)(lg + TG * E);
  int* cnt = ids_l + TG * topk;
  for (int i = blockIdx.x * 512 + threadIdx.x; i < cap; i += gridDim.x * 512) sorted_token[i] = -1;
  for (int e = threadIdx.x; e < E; e += 512) cnt[e] = 0;
  token_logits<W, TG, 4, 512>(x, wr, shared_w, rows, E, logits, T, H, bias, xs, 0, 1);
  __syncthreads();
  if (wave < nt)
    select_token(logits + wave * rows, rows, E, topk, renorm, groups, keep, lg + wave * E, ids + (size_t)(t0 + wave) * topk, ids_l + wave * topk,
                 weights + (size_t)(t0 + wave) * topk, shared_gate + t0 + wave, correction, n_real, wscale);
  __syncthreads();
  if (wave) return;
  int my_e, my_rank;
  rank_segment(ids_l, 0, nt * topk, E, cnt, pair_slot + (size_t)t0 * topk, false, my_e, my_rank);
  __builtin_amdgcn_wave_barrier();
  for (int e = threadIdx.x; e < E; e += TQ_WAVE) table[(size_t)blockIdx.x * E + e] = cnt[e];
}

// per: segments of a workgroup; seg: pairs of a segment.  LDS: [2][C][E] sums, [E] first rows, [per][E] a segment's first rows.
#define RP 1024      // threads
__global__ __launch_bounds__(RP) void route_place_kernel(const int* __restrict__ ids, int n_pairs, int E, int topk, int V, int per, int seg,
                                                         const int* __restrict__ table, int unit, int per_item, int cap,
                                                         int* __restrict__ sorted_token, int* __restrict__ pair_slot,
                                                         int* __restrict__ tile_expert, int* __restrict__ n_tiles, int n_real) {
  extern __shared__ int sm_p[];
  const int C = RP / E, v0 = blockIdx.x * per, v1 = min(v0 + per, V), n = v1 - v0;
  int* all = sm_p;
  int* before = all + C * E;
  int* starts = before + C * E;
  int* first = starts + E;
  for (int idx = threadIdx.x; idx < n * E; idx += RP) first[idx] = table[(size_t)v0 * E + idx];
  for (int idx = threadIdx.x; idx < C * E; idx += RP) {      // thread (c, e): segments c, c + C, ..
    const int c = idx / E, e = idx % E;
    int sum = 0, mine = 0;
    for (int v = c; v < V; v += 8 * C) {
      int t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = table[(size_t)min(v + u * C, V - 1) * E + e];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        sum += v + u * C < V ? t[u] : 0;
        mine += v + u * C < v0 ? t[u] : 0;
      }
    }
    all[idx] = sum;
    before[idx] = mine;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += RP) {
    int total = 0, mine = 0;
    for (int c = 0; c < C; ++c) {
      total += all[c * E + e];
      mine += before[c * E + e];
    }
    starts[e] = e < n_real ? (total + unit - 1) / unit * unit : 0;
    for (int s = 0; s < n; ++s) {
      const int c = first[s * E + e];
      first[s * E + e] = mine;
      mine += c;
    }
  }
  __syncthreads();
  if (threadIdx.x / TQ_WAVE == 0) scan_starts(starts, E, unit, per_item, cap, tile_expert, n_tiles, blockIdx.x == 0);
  __syncthreads();
  const int beg = v0 * seg, end = min(v1 * seg, n_pairs);
  for (int i = beg + threadIdx.x; i < end; i += RP) {
    const int e = ids[i], r = starts[e] + first[(i - beg) / seg * E + e] + pair_slot[i];
    pair_slot[i] = e < n_real ? r : -1;
    if (e < n_real) sorted_token[r] = i / topk;
  }
}

// The same order by several workgroups, for steps of many tokens (one workgroup's waves go through 32,768 pairs in
// 56 us, a compute unit's instructions being what it takes): three launches over V = 16 * workgroups waves that own
// the pairs in V contiguous runs, as the waves of the one workgroup do.  count: every wave ranks its pairs and leaves
// its counts per expert in table[v][e]; scan (one workgroup): the counts become each wave's first row within its
// expert, table[V][e] each expert's first row, and the row tiles and items are written; place: every pair's row.
// The results are those of the one workgroup: pairs in order of expert and, within an expert, of pair.
// table: (V + 1) * E ints of memory.
#define AC 8      // waves whose counts one thread of the scan adds up
__global__ __launch_bounds__(64 * AW) void align_count_kernel(const int* __restrict__ ids, int n_pairs, int E, int cap,
                                                              int* __restrict__ sorted_token,
                                                              int* __restrict__ pair_slot, int* __restrict__ table) {
  extern __shared__ int cnt[];       // [AW][E]
  const int wave = threadIdx.x / TQ_WAVE, lane = threadIdx.x % TQ_WAVE;
  const int V = gridDim.x * AW, v = blockIdx.x * AW + wave;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < cap; i += gridDim.x * blockDim.x) sorted_token[i] = -1;
  for (int i = threadIdx.x; i < AW * E; i += blockDim.x) cnt[i] = 0;
  __syncthreads();
  const int per = ((n_pairs + V - 1) / V + TQ_WAVE - 1) / TQ_WAVE * TQ_WAVE;
  const int seg_beg = min(n_pairs, v * per), seg_end = min(n_pairs, seg_beg + per);
  int my_e = -1, my_rank = 0;
  rank_segment(ids, seg_beg, seg_end, E, cnt + wave * E, pair_slot, false, my_e, my_rank);
  __builtin_amdgcn_wave_barrier();
  for (int e = lane; e < E; e += TQ_WAVE) table[(size_t)v * E + e] = cnt[wave * E + e];
}

__global__ __launch_bounds__(64 * AW) void align_scan_kernel(int* __restrict__ table, int V, int E, int unit, int per_item, int cap,
                                                             int* __restrict__ tile_expert, int* __restrict__ n_tiles,
                                                             int n_real) {
  extern __shared__ int sm_a[];        // [chunks][E] sums of AC waves' counts, then E starts
  const int chunks = (V + AC - 1) / AC;
  int* starts = sm_a + chunks * E;
  // thread (chunk c, expert e): the counts of waves AC c .. AC c + AC - 1, all asked for at once
  for (int idx = threadIdx.x; idx < chunks * E; idx += blockDim.x) {
    const int c = idx / E, e = idx % E;
    int sum = 0;
#pragma unroll
    for (int u = 0; u < AC; ++u) sum += AC * c + u < V ? table[(size_t)(AC * c + u) * E + e] : 0;
    sm_a[idx] = sum;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int total = 0;
    for (int c = 0; c < chunks; ++c) {
      const int t = sm_a[c * E + e];
      sm_a[c * E + e] = total;
      total += t;
    }
    starts[e] = e < n_real ? (total + unit - 1) / unit * unit : 0;
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < chunks * E; idx += blockDim.x) {
    const int c = idx / E, e = idx % E;
    int cv[AC];
#pragma unroll
    for (int u = 0; u < AC; ++u) cv[u] = AC * c + u < V ? table[(size_t)(AC * c + u) * E + e] : 0;
    int total = sm_a[idx];
#pragma unroll
    for (int u = 0; u < AC; ++u)
      if (AC * c + u < V) {
        table[(size_t)(AC * c + u) * E + e] = total;
        total += cv[u];
      }
  }
  if (threadIdx.x / TQ_WAVE == 0) scan_starts(starts, E, unit, per_item, cap, tile_expert, n_tiles);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) table[(size_t)V * E + e] = starts[e];
}

__global__ __launch_bounds__(64 * AW) void align_place_kernel(const int* __restrict__ ids, int n_pairs, int E, int topk,
                                                              const int* __restrict__ table,
                                                              int* __restrict__ pair_slot,
                                                              int* __restrict__ sorted_token, int n_real) {
  extern __shared__ int sm_a[];        // [AW][E] first rows of this workgroup's waves within the experts, then E starts
  const int wave = threadIdx.x / TQ_WAVE, lane = threadIdx.x % TQ_WAVE;
  const int V = gridDim.x * AW, v = blockIdx.x * AW + wave;
  for (int i = threadIdx.x; i < AW * E; i += blockDim.x) sm_a[i] = table[(size_t)blockIdx.x * AW * E + i];
  for (int e = threadIdx.x; e < E; e += blockDim.x) sm_a[AW * E + e] = table[(size_t)V * E + e];
  __syncthreads();
  const int* off = sm_a + wave * E;
  const int* starts = sm_a + AW * E;
  const int per = ((n_pairs + V - 1) / V + TQ_WAVE - 1) / TQ_WAVE * TQ_WAVE;
  const int seg_beg = min(n_pairs, v * per), seg_end = min(n_pairs, seg_beg + per);
  for (int i0 = seg_beg + lane; i0 < seg_end; i0 += 4 * TQ_WAVE) {
    int e[4], rk[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * TQ_WAVE;
      e[u] = i < seg_end ? ids[i] : 0;
      rk[u] = i < seg_end ? pair_slot[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * TQ_WAVE;
      if (i < seg_end && e[u] >= n_real) {
        pair_slot[i] = -1;
      } else if (i < seg_end) {
        const int r = starts[e[u]] + off[e[u]] + rk[u];
        pair_slot[i] = r;
        sorted_token[r] = i / topk;
      }
    }
  }
}

// Workgroups for the order of n_pairs pairs by several workgroups, or 0: the one workgroup does it (few pairs, or
// more experts than the scan's LDS holds, or a table too small).  Measured with 60 experts, 4 per token: 8,192 pairs
// 12 us against 17, 32,768 pairs 15 against 56, 131,072 pairs 40 against 225; 4,096 pairs 9 against 8.
#define ALIGN_MULTI_FROM 8192
static int align_workgroups(int n_pairs, int E, size_t table_ints) {
  if (n_pairs < ALIGN_MULTI_FROM) return 0;
  int g = n_pairs / 1024;
  g = g < 2 ? 2 : (g > 16 ? 16 : g);
  const int V = g * AW, chunks = (V + AC - 1) / AC;
  if ((size_t)(V + 1) * E > table_ints) return 0;
  if (((size_t)(chunks + 1) * E + 0) * sizeof(int) > 64 * 1024 || (size_t)(AW + 1) * E * sizeof(int) > 64 * 1024) return 0;
  return g;
}

static int launch_align_multi(const int* ids, int n_pairs, int E, int topk, int unit, int per_item, int cap, int* sorted_token,
                              int* pair_slot, int* tile_expert, int* n_tiles, int* table, int g, hipStream_t st,
                              int n_real = 1 << 30) {
  const int V = g * AW, chunks = (V + AC - 1) / AC;
  const size_t lds_count = (size_t)AW * E * sizeof(int), lds_scan = (size_t)(chunks + 1) * E * sizeof(int),
               lds_place = (size_t)(AW + 1) * E * sizeof(int);
  if (lds_scan > 48 * 1024)
    (void)hipFuncSetAttribute((const void*)align_scan_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_scan);
  if (lds_place > 48 * 1024) {
    (void)hipFuncSetAttribute((const void*)align_count_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_place);
    (void)hipFuncSetAttribute((const void*)align_place_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_place);
  }
  hipLaunchKernelGGL(align_count_kernel, dim3(g), dim3(64 * AW), lds_count, st, ids, n_pairs, E, cap, sorted_token,
                     pair_slot, table);
  hipLaunchKernelGGL(align_scan_kernel, dim3(1), dim3(64 * AW), lds_scan, st, table, V, E, unit, per_item, cap, tile_expert,
                     n_tiles, n_real);
  hipLaunchKernelGGL(align_place_kernel, dim3(g), dim3(64 * AW), lds_place, st, ids, n_pairs, E, topk, table, pair_slot,
                     sorted_token, n_real);
  TQ_LAUNCH_CHECK();
  return 0;
}

// The choice and the order of pairs in one workgroup of NW waves, for up to NW tokens (decoding): wave w chooses for token w,
// then all waves order the pairs; the same device functions and so the same results as the two kernels.
template <int NW>
__global__ __launch_bounds__(64 * NW) void select_align_kernel(const float* __restrict__ logits, int rows, int E,
                                                               int topk, int renorm, int groups, int keep,
                                                               int* __restrict__ ids, float* __restrict__ weights,
                                                               float* __restrict__ shared_gate, int T, int unit,
                                                               int per_item, int cap, int* __restrict__ sorted_token,
                                                               int* __restrict__ pair_slot,
                                                               int* __restrict__ tile_expert,
                                                               int* __restrict__ n_tiles,
                                                               const float* __restrict__ correction, int n_real,
                                                               float wscale) {
  extern __shared__ int sm_i[];       // (NW + 1) * E ints for the order, NW * topk ids, NW * E floats for the choice
  if constexpr (NW == 1) {
    // One token whose experts fit the lanes: a chosen expert has one row, the first of its unit, and its place among the units is the
    // number of chosen experts below it.
    const int lane = threadIdx.x;
    if (int e; choose_small(logits, rows, E, topk, renorm, groups, keep, weights, shared_gate, correction, n_real, wscale, e)) {
      unsigned long long lo = 0, hi = 0;      // (an expert twice only where fewer than topk logits are finite: the general order below)
      for (int k = 0; k < topk; ++k) {
        const int c = __builtin_amdgcn_readlane(e, k);
        (c < 64 ? lo : hi) |= 1ull << (c & 63);
      }
      if (lane < topk) ids[lane] = e;
      if (__popcll(lo) + __popcll(hi) == topk) {
        lo &= n_real < 64 ? (1ull << n_real) - 1ull : ~0ull;
        hi &= n_real <= 64 ? 0ull : n_real < 128 ? (1ull << (n_real - 64)) - 1ull : ~0ull;
        const int n = __popcll(lo) + __popcll(hi);
        if (lane < topk) {
          const unsigned long long below = (1ull << (e & 63)) - 1ull;
          const int place = e < 64 ? __popcll(lo & below) : __popcll(lo) + __popcll(hi & below);
          pair_slot[lane] = e < n_real ? place * unit : -1;
          if (e < n_real) {
            tile_expert[place] = e;
            tile_expert[cap / unit + place] = place;
          }
        }
        for (int i = lane; i < cap; i += TQ_WAVE) sorted_token[i] = i < n * unit && i % unit == 0 ? 0 : -1;
        if (clear_queues(n_tiles, per_item) && lane == 0) n_tiles[2] = n;
        if (lane == 0) n_tiles[0] = n_tiles[1] = n;
        return;
      }
      if (lane < topk) sm_i[lane] = e;
      __syncthreads();
      align_pairs<NW>(sm_i, topk, E, topk, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, sm_i + topk, n_real);
      return;
    }
  }
  int* cnt = sm_i;
  int* ids_l = cnt + (NW + 1) * E;
  float* lg = (float*)(ids_l + NW * topk);
  const int wave = threadIdx.x / TQ_WAVE;
  if (wave < T)
    select_token(logits + (size_t)wave * rows, rows, E, topk, renorm, groups, keep, lg + wave * E, ids + (size_t)wave * topk,
                 ids_l + wave * topk, weights + (size_t)wave * topk, shared_gate + wave, correction, n_real, wscale);
  __syncthreads();
  align_pairs<NW>(ids_l, T * topk, E, topk, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, cnt, n_real);
}

// Row tiles that an item holds at most, with TQ_WITH_QUEUES where there are queues to zero; takes TQ_ITEMS_OF_FOUR and TQ_ORDER_QUEUES
// off `unit`.
static int units_per_item(int& unit) {
  int per_item = 2;
  if (unit == 64 + TQ_ORDER_QUEUES || unit == 64 + TQ_ITEMS_OF_FOUR + TQ_ORDER_QUEUES) unit -= TQ_ORDER_QUEUES, per_item += TQ_WITH_QUEUES;
  if (unit >= TQ_ITEMS_OF_FOUR) unit -= TQ_ITEMS_OF_FOUR, per_item += 2;
  return per_item;
}

// cap: rows that sorted_token holds, a multiple of unit and at least n_pairs + min(E, n_pairs) * (unit - 1);
// tile_expert holds 2 * cap / unit entries (row tiles, then items), n_tiles two.
static int moe_align_impl(const int* ids, int n_pairs, int E, int topk, int unit, int per_item, int cap, int* sorted_token,
                          int* pair_slot, int* tile_expert, int* n_tiles, hipStream_t st, int n_real) {
  if (n_pairs <= 0) return 0;
  if (unit < 1 || cap % unit != 0 || cap < n_pairs + (E < n_pairs ? E : n_pairs) * (unit - 1)) return TQ_ERR_BAD_ARG;
  const size_t shmem = (size_t)(AW + 1) * E * sizeof(int);
  if (shmem > 160 * 1024) return TQ_ERR_UNSUPPORTED;
  if (shmem > 48 * 1024)
    (void)hipFuncSetAttribute((const void*)moe_align_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(64 * AW), shmem, st, ids, n_pairs, E, topk, unit, per_item, cap,
                     sorted_token, pair_slot, tile_expert, n_tiles, n_real);
  TQ_LAUNCH_CHECK();
  return 0;
}

TQ_API int tq_moe_align(const int* ids, int n_pairs, int E, int topk, int unit, int cap, int* sorted_token,
                        int* pair_slot, int* tile_expert, int* n_tiles, hipStream_t st) {
  const int per_item = units_per_item(unit);
  return moe_align_impl(ids, n_pairs, E, topk, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, st, E);
}

// Whether the choice and the order go in two launches by many workgroups, and how: tg tokens to a workgroup of route_choose, V of those, per
// of its segments to a workgroup of route_place.  What the launches saved and the order by many workgroups gain must be more than every
// workgroup's own way through all rows of wr and the table of V counts per expert costs (us apart and this way; of 800 sizes drawn the way taken is
// more than 4 % slower than the other form in 8, and 1.19 times as fast in the geometric mean):
//  * rows of up to 5,120, of which router_logits has 8 tokens to a workgroup too:
//    - 8 experts and more, fewer leaving most waves without rows (929 tokens, 5 of 4,096, one a token 13.0 and 16.6; 12,630, 3 of 2,560, two 55 and
//      67), and up to 8 for every pair of a workgroup's, the table's way (1,145, 160 of 5,120, one 61 and 84; 1,210, 384 of 2,560, one 63 and 86; 512, 120
//      of 3,584, four 24.5 and 27.8; 1,024, 128 of 1,024, one 16.4 and 19.1; but 1,500, 120 of 3,072, four 54 and 39), 6 with rows beyond 4,608 (512,
//      96 of 5,120, four 28.5 and 29.3);
//    - pairs whose order takes one workgroup some time (1,181, 8 of 3,072, two 15.0 and 16.5, 671, 17 of 1,000, one 10.6 and 11.5; 1,500, 8 of
//      3,072, four 27.3 and 18.0, 906, 16 of 1,536, eight 21.9 and 14.1), or 16 experts of rows beyond 2,560, of which router_logits has a workgroup to
//      a unit (868, 32 of 3,072, two 24.1 and 14.0);
//    - not beyond 4,608 from 3,072 tokens on (5,120: 3,000 tokens of 16 experts 50 and 43, 4,096 52 and 53; of 8 44 and 49, of 32 64 and 74), 1,025 beyond
//      128 experts (1,341 of 160, eight 81 and 95), nor between
//      2,048 and 2,560 from 7,169 on (6,743 of 24, two 46 and 43; 13,980 of 16, four 70 and 77), which have half as many tokens to a workgroup here as
//      there; nor with more than 192 experts just beyond 1,024 tokens, which leave half the units idle (1,115, 256 of 2,048, six 53 and 56; 1,220, 384
//      of 3,072, six 95 and 100; 1,429, 359 of 2,560, six 89 and 79);
//  * longer rows, of which router_logits has few tokens to a workgroup, from 10 experts on, 16 where there are fewer than 4 here (1,024, 249 of 6,144,
//    four 196 and 86; 859, 10 of 8,192, six 35 and 23; 512, 33 of 10,240, one 34 and 26; but 1,280, 8 of 10,240, eight 40 and 46);
//  * 512 tokens (1,024 beyond 128 experts): fewer leave compute units idle, over which the other form deals the rows of wr (60 experts, 200 tokens
//    12.8 and 14.7, 400 15.7 and 15.6; 256, 401 35.5 and 41.0, 700 44.6 and 45.2, 1,024 48.9 and 46.3); a table of up to 65,536 counts (256 experts,
//    2,048 tokens, 65,536 counts, 78 and 63, 3,001 tokens, 96,256, 108 and 111, 8,192, 262,144, 191 and 224).
struct RouteMany {
  int tg, V, per;
  size_t lds;
};
static bool route_many_suits(int T, int E, int rows, int topk, int H, RouteMany* r) {
  if (T < (E <= 128 ? 512 : 1024)) return false;
  const size_t hp = ((size_t)H + 511) / 512 * 512;
  auto lds = [&](int tg) { return (tg * (hp + rows + E + topk) + E) * 4; };
  // So few tokens to a workgroup that there is one to a compute unit while they last, and where there are more, that two share one.
  int tg = T <= 512 ? 2 : T <= 1024 ? 4 : 8;
  while (tg > 1 && lds(tg) > (T > 2048 ? 80 : 160) * 1024) tg /= 2;
  const int V = (T + tg - 1) / tg;
  if (lds(tg) > 160 * 1024 || (int64_t)V * E > 65536) return false;
  if (hp <= 5120) {
    const bool tall = hp > 4608;
    if (E < 8 || E > (tall ? 6 : 8) * tg * topk || (E > 192 && T > 1024 && T < 1408)) return false;
    if ((int64_t)T * topk < (E < 10 ? 2560 : 2048) && (hp <= 2560 || E < 16)) return false;
    if (tall ? T >= (E > 128 ? 1025 : 3072) : hp > 2048 && hp <= 2560 && T > 7168) return false;
  } else if (E < (tg < 4 ? 16 : 10)) {
    return false;
  }
  const int even = (V + 63) / 64;
  *r = {tg, V, even < 16 ? 16 : even, lds(tg)};
  return true;
}
TQ_API int tq_route_in_two(int T, int E, int shared, int topk, int H) {
  RouteMany r;
  return E > 0 && topk > 0 && H > 0 && route_many_suits(T, E, E + (shared ? 1 : 0), topk, H, &r);
}
// table: T * E ints.
static int route_many(const RouteMany& r, const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E, int topk,
                      int renorm, int groups, int keep, int* ids, float* weights, float* shared_gate, int* table, int unit, int per_item, int cap,
                      int* sorted_token, int* pair_slot, int* tile_expert, int* n_tiles, int T, int H, hipStream_t st,
                      const float* correction, int n_real, float wscale) {
  if (topk < 1 || topk > 64 || topk > E || E > 8192) return TQ_ERR_UNSUPPORTED;
  const int rows = E + (shared_w ? 1 : 0), n_pairs = T * topk, tg = r.tg, V = r.V, per = r.per;
  if (unit < 1 || cap % unit != 0 || cap < n_pairs + (E < n_pairs ? E : n_pairs) * (unit - 1)) return TQ_ERR_BAD_ARG;
  const size_t shmem = r.lds;
  // (V E <= 65,536 and T / V <= 8 leave at most 508 experts, and route_place 42,672 bytes of LDS)
  const size_t lds_place = ((size_t)(2 * (RP / E) + 1 + per) * E) * sizeof(int);
#define TQ_CHOOSE(TGV)                                                                                                                    \
  do {                                                                                                                                    \
    if (shmem > 48 * 1024)                                                                                                                \
      (void)hipFuncSetAttribute((const void*)route_choose_kernel<W, TGV>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem); \
    hipLaunchKernelGGL((route_choose_kernel<W, TGV>), dim3(V), dim3(512), shmem, st, x, (const W*)wr, (const W*)shared_w, rows, E, T, \
                       H, bias, topk, renorm, groups, keep, correction, n_real, wscale, ids, weights, shared_gate, cap, sorted_token, \
                       pair_slot, table);                                                                                                 \
  } while (0)
  TQ_DISPATCH_W(wtype, {
    if (tg == 8) TQ_CHOOSE(8);
    else if (tg == 4) TQ_CHOOSE(4);
    else if (tg == 2) TQ_CHOOSE(2);
    else TQ_CHOOSE(1);
  });
#undef TQ_CHOOSE
  hipLaunchKernelGGL(route_place_kernel, dim3((V + per - 1) / per), dim3(RP), lds_place, st, ids, n_pairs, E, topk, V, per, tg * topk, table, unit,
                     per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, n_real);
  TQ_LAUNCH_CHECK();
  return 0;
}

// tq_router_topk followed by tq_moe_align, with the same results: up to 16 tokens in two launches, many as route_many_suits says in two others,
// else in three, or five where several workgroups order the pairs (from 8,192 on).  logits: scratch of T * (E + 1) floats (T * E without a shared
// gate vector); what it holds afterwards means nothing.
// groups, keep: the choice within the best `keep` of `groups` groups of experts (1, 1: among all).
static int route_impl(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E,
                      int topk, int renorm, int groups, int keep, int* ids, float* weights, float* shared_gate,
                      float* logits, int unit, int cap, int* sorted_token, int* pair_slot, int* tile_expert,
                      int* n_tiles, int T, int H, hipStream_t st, const float* correction, int n_real, float wscale = 1.0f) {
  if (T <= 0) return 0;
  const int per_item = units_per_item(unit);
  if (!groups_ok(E, topk, groups, keep)) return TQ_ERR_BAD_ARG;
  const size_t shmem = ((size_t)(AW + 1) * E + (size_t)AW * topk + (size_t)AW * E) * 4;
  if (T > AW || shmem > 64 * 1024) {
    RouteMany r;
    if (route_many_suits(T, E, E + (shared_w ? 1 : 0), topk, H, &r))
      return route_many(r, x, wr, shared_w, bias, wtype, E, topk, renorm, groups, keep, ids, weights, shared_gate, (int*)logits, unit, per_item, cap,
                        sorted_token, pair_slot, tile_expert, n_tiles, T, H, st, correction, n_real, wscale);
    const int rc = router_topk_impl(x, wr, shared_w, bias, wtype, E, topk, renorm, groups, keep, ids, weights,
                                    shared_gate, logits, T, H, st, correction, n_real, wscale);
    if (rc) return rc;
    // once the experts are chosen the logits are done with: the order by several workgroups keeps its table there
    const int n = T * topk;
    const int g = align_workgroups(n, E, (size_t)T * (E + (shared_w ? 1 : 0)));
    if (g == 0) return moe_align_impl(ids, n, E, topk, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, st, n_real);
    if (unit < 1 || cap % unit != 0 || cap < n + (E < n ? E : n) * (unit - 1)) return TQ_ERR_BAD_ARG;
    return launch_align_multi(ids, n, E, topk, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles, (int*)logits, g,
                              st, n_real);
  }
  if (topk < 1 || topk > 64 || topk > E || E > 8192) return TQ_ERR_UNSUPPORTED;
  const int n_pairs = T * topk;
  if (unit < 1 || cap % unit != 0 || cap < n_pairs + (E < n_pairs ? E : n_pairs) * (unit - 1)) return TQ_ERR_BAD_ARG;
  const int rc = launch_router_logits(x, wr, shared_w, wtype, E, logits, T, H, st, bias);
  if (rc) return rc;
  if (T == 1) {      // one wave: its barriers cost nothing
    const size_t shmem1 = ((size_t)2 * E + topk + E) * 4;
    hipLaunchKernelGGL(select_align_kernel<1>, dim3(1), dim3(64), shmem1, st, logits, E + (shared_w ? 1 : 0), E, topk,
                       renorm, groups, keep, ids, weights, shared_gate, T, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles,
                       correction, n_real, wscale);
    TQ_LAUNCH_CHECK();
    return 0;
  }
  if (shmem > 48 * 1024)
    (void)hipFuncSetAttribute((const void*)select_align_kernel<AW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
  hipLaunchKernelGGL(select_align_kernel<AW>, dim3(1), dim3(64 * AW), shmem, st, logits, E + (shared_w ? 1 : 0), E, topk,
                     renorm, groups, keep, ids, weights, shared_gate, T, unit, per_item, cap, sorted_token, pair_slot, tile_expert, n_tiles,
                       correction, n_real, wscale);
  TQ_LAUNCH_CHECK();
  return 0;
}

TQ_API int tq_route_biased(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E,
                           int topk, int renorm, int groups, int keep, int* ids, float* weights, float* shared_gate,
                           float* logits, int unit, int cap, int* sorted_token, int* pair_slot, int* tile_expert,
                           int* n_tiles, int T, int H, hipStream_t st) {
  return route_impl(x, wr, shared_w, bias, wtype, E, topk, renorm, groups, keep, ids, weights, shared_gate, logits, unit, cap,
                    sorted_token, pair_slot, tile_expert, n_tiles, T, H, st, nullptr, E);
}

// A router whose softmax runs over all E rows, whose choice is by score + correction[e] and whose weights are the scores
// themselves, not renormalised.  The rows from n_real on are experts without matrices (the identity): their pairs get
// pair_slot -1 and no rows, and id_gate[t] (null if n_real == E) is the sum of the token's weights for them.
TQ_API int tq_route_scored(const float* x, const void* wr, const float* correction, int wtype, int E, int n_real, int topk,
                           int* ids, float* weights, float* id_gate, float* logits, int unit, int cap, int* sorted_token,
                           int* pair_slot, int* tile_expert, int* n_tiles, int T, int H, hipStream_t st) {
  if (n_real < 1 || n_real > E || (n_real < E && !id_gate) || !correction) return TQ_ERR_BAD_ARG;
  return route_impl(x, wr, nullptr, nullptr, wtype, E, topk, 0, 1, 1, ids, weights, id_gate, logits, unit, cap, sorted_token,
                    pair_slot, tile_expert, n_tiles, T, H, st, correction, n_real);
}

TQ_API int tq_route_grouped(const float* x, const void* wr, const void* shared_w, int wtype, int E, int topk, int renorm,
                            int groups, int keep, int* ids, float* weights, float* shared_gate, float* logits, int unit,
                            int cap, int* sorted_token, int* pair_slot, int* tile_expert, int* n_tiles, int T, int H,
                            hipStream_t st) {
  return tq_route_biased(x, wr, shared_w, nullptr, wtype, E, topk, renorm, groups, keep, ids, weights, shared_gate, logits,
                         unit, cap, sorted_token, pair_slot, tile_expert, n_tiles, T, H, st);
}

TQ_API int tq_route(const float* x, const void* wr, const void* shared_w, int wtype, int E, int topk, int renorm,
                    int* ids, float* weights, float* shared_gate, float* logits, int unit, int cap, int* sorted_token,
                    int* pair_slot, int* tile_expert, int* n_tiles, int T, int H, hipStream_t st) {
  return tq_route_grouped(x, wr, shared_w, wtype, E, topk, renorm, 1, 1, ids, weights, shared_gate, logits, unit, cap,
                          sorted_token, pair_slot, tile_expert, n_tiles, T, H, st);
}

// A router whose experts' scores are the sigmoids of their logits (bias: added to the logits first): the `topk` largest
// scores, within the best `keep` of `groups` groups (1, 1: among all), whose score is their largest score or, with
// pair_groups, the sum of their two largest; the weights are the chosen scores over (their sum + 1e-20), times wscale.
TQ_API int tq_router_topk_sigmoid(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E,
                                  int topk, int groups, int keep, int pair_groups, float wscale, int* ids, float* weights,
                                  float* shared_gate, float* logits, int T, int H, hipStream_t st) {
  return router_topk_impl(x, wr, shared_w, bias, wtype, E, topk, TQ_ROUTE_SIGMOID | (pair_groups ? TQ_ROUTE_PAIR_GROUPS : 0),
                          groups, keep, ids, weights, shared_gate, logits, T, H, st, nullptr, E, wscale);
}

TQ_API int tq_route_sigmoid(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E, int topk,
                            int groups, int keep, int pair_groups, float wscale, int* ids, float* weights, float* shared_gate,
                            float* logits, int unit, int cap, int* sorted_token, int* pair_slot, int* tile_expert, int* n_tiles,
                            int T, int H, hipStream_t st) {
  return route_impl(x, wr, shared_w, bias, wtype, E, topk, TQ_ROUTE_SIGMOID | (pair_groups ? TQ_ROUTE_PAIR_GROUPS : 0), groups,
                    keep, ids, weights, shared_gate, logits, unit, cap, sorted_token, pair_slot, tile_expert, n_tiles, T, H, st,
                    nullptr, E, wscale);
}

// A router whose weights are the softmax over the chosen experts' logits, times wscale (bias: added to the logits first).
TQ_API int tq_router_topk_weighted(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E,
                                   int topk, int groups, int keep, float wscale, int* ids, float* weights, float* shared_gate,
                                   float* logits, int T, int H, hipStream_t st) {
  return router_topk_impl(x, wr, shared_w, bias, wtype, E, topk, 1, groups, keep, ids, weights, shared_gate, logits, T, H, st,
                          nullptr, E, wscale);
}

TQ_API int tq_route_weighted(const float* x, const void* wr, const void* shared_w, const float* bias, int wtype, int E, int topk,
                             int groups, int keep, float wscale, int* ids, float* weights, float* shared_gate, float* logits,
                             int unit, int cap, int* sorted_token, int* pair_slot, int* tile_expert, int* n_tiles, int T, int H,
                             hipStream_t st) {
  return route_impl(x, wr, shared_w, bias, wtype, E, topk, 1, groups, keep, ids, weights, shared_gate, logits, unit, cap,
                    sorted_token, pair_slot, tile_expert, n_tiles, T, H, st, nullptr, E, wscale);
}
