// Online-softmax pooling of one compressed entry: a lane folds tokens of 8
// consecutive channels into (max, sum of weights, weighted sum), and the
// lanes that folded different tokens of the same channels are merged.
// Pooling of a block of m tokens (TokenLevelCompressor, csa.py:81-87):
//   v_i = z_i + bias_i ; out = sum_i exp(v_i) c_i / sum_i exp(v_i)
#pragma once

#include "skv_entry.h"

namespace skv {

constexpr int kPoolWave = 64;
constexpr int kMaxGroups = 4;  // channels <= 64*8*4 = 2048

struct PoolLane {
  float mx[8], sum[8], acc[8];
};

__device__ __forceinline__ void pool_reset(PoolLane& st) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    st.mx[j] = -INFINITY;
    st.sum[j] = 0.f;
    st.acc[j] = 0.f;
  }
}

// The weight exp(v - M) of value v against the running max M >= v (NaN when
// any value was one).  Where v - M is NaN the weight is 1: a value of -inf
// counts until a finite one arrives and takes its weight to 0, in any order,
// and pool_out turns a block that is -inf throughout, or holds several +inf or
// a NaN, into NaN, as a softmax does.  x log2(e) is carried in two floats, which
// keeps the sums as close to the 64-bit ones as a library exp (one float
// costs 4% at 4 tokens) in a third of its instructions; below e^-104 it is 0.
__device__ __forceinline__ float pool_weight(float v, float M) {
  constexpr float kLog2e = 1.44269504088896341f, kLn2 = 0.693147180559945309f;
  const float x = fmaxf(fminf(v - M, 0.f), -104.f);
  const float t = x * kLog2e;
  const float r = fmaf(x, kLog2e, -t);
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, r * kLn2, e);
}

// Folds N tokens (values v, rows c) into the state.
template <int N>
__device__ __forceinline__ void pool_fold(PoolLane& st, const float (&v)[N][8], const float (&c)[N][8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float M = st.mx[j];
#pragma unroll
    for (int u = 0; u < N; ++u) M = __builtin_elementwise_maximum(M, v[u][j]);  // NaN stays
    const float s = pool_weight(st.mx[j], M);
    float sum = st.sum[j] * s, acc = st.acc[j] * s;
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const float w = pool_weight(v[u][j], M);
      sum += w;
      acc = fmaf(w, c[u][j], acc);
    }
    st.mx[j] = M;
    st.sum[j] = sum;
    st.acc[j] = acc;
  }
}

// Folds one token (values v, rows c).  Appends and decode steps fold with it in
// turn, so that a state which one of them leaves means the same to the other.
// Where v - max is NaN the weight is 1, as in pool_weight.
__device__ __forceinline__ void pool_fold_token(PoolLane& st, const float (&v)[8], const float (&c)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float d = v[j] - st.mx[j];
    const bool up = v[j] > st.mx[j];
    const float t = d != d ? 1.f : expf(-__builtin_fabsf(d));  // rescales the state, or weighs the token
    st.sum[j] = fmaf(t, up ? st.sum[j] : 1.f, up ? 1.f : st.sum[j]);
    st.acc[j] = fmaf(t, up ? st.acc[j] : c[j], up ? c[j] : st.acc[j]);
    st.mx[j] = __builtin_elementwise_maximum(st.mx[j], v[j]);  // NaN stays
  }
}

// Folds N tokens one after another, as decode steps do: the same sums whether a
// block comes at once or a token at a time (the codes of fp8 entries hang on their
// last bits).
template <int N>
__device__ __forceinline__ void pool_fold_serial(PoolLane& st, const float (&v)[N][8], const float (&c)[N][8]) {
#pragma unroll
  for (int u = 0; u < N; ++u) pool_fold_token(st, v[u], c[u]);
}

// The state of a lane's channels seen from the larger max M[j]: sums and
// weighted sums of several lanes can then be added.
__device__ __forceinline__ void pool_rebase(PoolLane& st, const float (&M)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float s = pool_weight(st.mx[j], M[j]);
    st.mx[j] = M[j];
    st.sum[j] *= s;
    st.acc[j] *= s;
  }
}

// The pooled value of channel j.
__device__ __forceinline__ float pool_out(const PoolLane& st, int j) {
  const float M = st.mx[j];
  const float q = st.acc[j] / st.sum[j];
  return (M != M) | (M == -INFINITY) | ((M == INFINITY) & (st.sum[j] > 1.f)) ? NAN : q;
}

}  // namespace skv
