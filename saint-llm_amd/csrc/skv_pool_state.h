// Online-softmax pooling of one compressed entry: a lane folds tokens, one
// after another, into its channels' (max, sum of weights, weighted sum).
// Pooling of a block of m tokens (TokenLevelCompressor, csa.py:81-87):
//   v_i = z_i + bias_i ; out = sum_i exp(v_i) c_i / sum_i exp(v_i)
#pragma once

#include "skv_entry.h"

namespace skv {

constexpr int kPoolWave = 64;
constexpr int kMaxGroups = 4;  // channels <= 64*8*4 = 2048

template <int kCh>
struct PoolLane {
  float mx[kCh], sum[kCh], acc[kCh];
};

template <int kCh>
__device__ __forceinline__ void pool_reset(PoolLane<kCh>& st) {
#pragma unroll
  for (int j = 0; j < kCh; ++j) {
    st.mx[j] = -INFINITY;
    st.sum[j] = 0.f;
    st.acc[j] = 0.f;
  }
}

// Folding one token (value v, row c) into a channel's state: exp(-|v - max|) rescales
// the state where v is above the max (up), otherwise it weighs the token.  Appends
// and decode steps all fold so, token by token in the sequence's order: an entry
// has the same bits whichever calls brought its tokens (the codes of fp8 entries
// hang on the last bits of the sums), and a state which one of them leaves means
// the same to the next.
// Where v - max is NaN the weight is 1: a value of -inf counts until a finite one
// arrives and takes its weight to 0, in any order, and pool_out turns a block that
// is -inf throughout, or holds several +inf or a NaN, into NaN, as a softmax does.
__device__ __forceinline__ float pool_weight(float v, float mx, bool& up) {
  const float d = v - mx;
  up = v > mx;
  return d != d ? 1.f : expf(-__builtin_fabsf(d));
}

__device__ __forceinline__ void pool_add(float& sum, float& acc, float w, bool up, float c) {
  sum = fmaf(sum, up ? w : 1.f, up ? 1.f : w);
  acc = fmaf(w, up ? acc : c, up ? c : acc);
}

__device__ __forceinline__ void pool_fold_token(PoolLane<8>& st, const float (&v)[8], const float (&c)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    bool up;
    const float w = pool_weight(v[j], st.mx[j], up);
    pool_add(st.sum[j], st.acc[j], w, up, c[j]);
    st.mx[j] = __builtin_elementwise_maximum(st.mx[j], v[j]);  // NaN stays
  }
}

// The pooled value of channel j.
__device__ __forceinline__ float pool_out(const PoolLane<8>& st, int j) {
  const float M = st.mx[j];
  const float q = st.acc[j] / st.sum[j];
  return (M != M) | (M == -INFINITY) | ((M == INFINITY) & (st.sum[j] > 1.f)) ? NAN : q;
}

}  // namespace skv
