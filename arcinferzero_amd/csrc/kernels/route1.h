// The routing of one token by one wave, shared by the kernels that route (reference zero/kernels/moe.cl:50-109): the NU
// largest of NE logits (ties: the lower expert), p = exp(l - max), weights p / sum of the selected p.  Lane k < NU
// returns the k-th choice and its weight.  NE <= 512.
#pragma once
#include "common.h"

#define ROUTE_PER_LANE 8

// A logit as an unsigned key in the order of the values: 0 for what no round picks (-inf, NaN), both zeros alike.
__device__ inline uint32_t route_key(float v) {
  const uint32_t u = __float_as_uint(v + 0.0f);
  return v > -INFINITY ? ((int)u < 0 ? ~u : u | 0x80000000u) : 0u;
}
__device__ inline float route_unkey(uint32_t k) {
  return k ? __uint_as_float((int)k < 0 ? k & 0x7FFFFFFFu : ~k) : -INFINITY;
}
// The wave's largest key, a scalar: six dependent maxima in the vector ALU (shifts inside the rows of 16 lanes, then each
// row's last lane into the rows behind it), read from the last lane.
__device__ inline uint32_t route_wave_max(uint32_t k) {
#define ROUTE_STEP(CTRL, ROWS) k = max(k, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k, CTRL, ROWS, 0xF, false));
  ROUTE_STEP(0x111, 0xF) ROUTE_STEP(0x112, 0xF) ROUTE_STEP(0x114, 0xF) ROUTE_STEP(0x118, 0xF)  // row_shr 1, 2, 4, 8
  ROUTE_STEP(0x142, 0xA) ROUTE_STEP(0x143, 0xC)                                                // row_bcast 15, 31
#undef ROUTE_STEP
  return (uint32_t)__builtin_amdgcn_readlane((int)k, 63);
}

// The reference's routing variants (zero/kernels/moe.cl:17-46), chosen per launch: escale (its -DESCALE, Gemma 4) -- each
// chosen expert's weight times escale[e] after the normalization; ebias (its -DROUTE_DS, DeepSeek-V4.1) -- the score is
// s = sqrt(softplus(logit)), experts are chosen by s + ebias[e], and the weights are s / (sum of the chosen s + 1e-20) *
// rscale.  Both null: the softmax routing.
struct RouteVariant {
  const float* escale = nullptr;
  const float* ebias = nullptr;
  float rscale = 1.0f;
};
__device__ inline float route_ds_sp(float g) { return sqrtf(g > 20.0f ? g + log1pf(expf(-g)) : log1pf(expf(g))); }

// The choices one after the other: the largest key of the wave, and of the lanes that hold it the lowest expert, by a
// ballot.  A round is a chain of about ten instructions -- with the (value, expert) pairs compared step by step, which it
// was, 60 -- and the exponentials are taken once at the end, lane k its own; their sum in the order of the choices.
// v: the lane's logits, of experts lane, lane + 64, .. (route_logits).
template <int PL>
__device__ inline void route_logits(const float* __restrict__ lg, int NE, int lane, float (&v)[PL]) {
#pragma unroll
  for (int i = 0; i < PL; ++i) v[i] = lg[min(i * 64 + lane, NE - 1)];
}
template <int PL>
__device__ inline void route_one_token_pl(const float (&v)[PL], const float* __restrict__ lg, int NE, int NU, int lane, int& sel, float& wt,
                                          const RouteVariant rv = RouteVariant()) {
  uint32_t key[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int e = i * 64 + lane;
    key[i] = e < NE ? route_key(rv.ebias ? route_ds_sp(v[i]) + rv.ebias[e] : v[i]) : 0u;
  }
  uint32_t mykey = 0, top = 0;
  int mysel = 0;
  for (int k = 0; k < NU; ++k) {
    uint32_t mine = key[0];
#pragma unroll
    for (int i = 1; i < PL; ++i) mine = max(mine, key[i]);
    const uint32_t m = route_wave_max(mine);
    int bi = NE - 1;  // (nothing left to pick: keep the index inside the tables)
    if (m) {
#pragma unroll
      for (int i = PL - 1; i >= 0; --i) {
        const uint64_t has = __ballot(key[i] == m);
        if (has) bi = i * 64 + __builtin_ctzll(has);
      }
    }
#pragma unroll
    for (int i = 0; i < PL; ++i)
      if (i * 64 + lane == bi) key[i] = 0;
    if (k == 0) top = m;
    if (lane == k) { mysel = bi; mykey = m; }
  }
  const float myp = rv.ebias ? (lane < NU ? route_ds_sp(lg[mysel]) : 0.0f) : expf(route_unkey(mykey) - route_unkey(top));
  float sum = 0.0f;
  for (int k = 0; k < NU; ++k) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myp), k));
  sel = mysel;
  wt = rv.ebias ? myp / (sum + 1e-20f) * rv.rscale : myp / sum;
  if (rv.escale) wt *= rv.escale[mysel];
}

// (two logits a lane serve up to 128 experts, the common case; the same steps either way)
template <int PL>
__device__ inline void route_one_token_of(const float* __restrict__ lg, int NE, int NU, int lane, int& sel, float& wt, const RouteVariant rv) {
  float v[PL];
  route_logits(lg, NE, lane, v);
  route_one_token_pl(v, lg, NE, NU, lane, sel, wt, rv);
}
__device__ inline void route_one_token(const float* __restrict__ lg, int NE, int NU, int lane, int& sel, float& wt,
                                       const RouteVariant rv = RouteVariant()) {
  if (NE <= 128) route_one_token_of<2>(lg, NE, NU, lane, sel, wt, rv);
  else route_one_token_of<ROUTE_PER_LANE>(lg, NE, NU, lane, sel, wt, rv);
}
// The shared expert's gate of a token (moe.cl:40, 46): sigmoid of the logit past the experts' when the row holds one;
// 1 with the -DROUTE_DS routing.
__device__ inline float route_sgate(const float* __restrict__ lg, int NE, bool has_gate, const RouteVariant rv) {
  return rv.ebias ? 1.0f : has_gate ? 1.0f / (1.0f + expf(-lg[NE])) : 0.0f;
}
