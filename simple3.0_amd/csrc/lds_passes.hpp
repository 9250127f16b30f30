// lds_passes.hpp - compile-time-size FFT passes in LDS (the pre-processing stages' row and column
// transforms): the ring length and the transforms per work-group are template constants, so every
// index, radix and loop bound folds at compile time.
#pragma once
#include "fft_lds.hpp"

namespace pfk {

// Radix order: one 4 first, the remaining factors in descending order
__host__ __device__ constexpr FftPlan make_fused_plan(int n) {
  FftPlan p = make_plan(n);
  if (p.np < 2 || n % 4 != 0) return p;
  FftPlan q{0, {0}};
  q.r[q.np++] = 4;
  int rest[16] = {0};
  int nr = 0;
  bool dropped = false;
  for (int i = 0; i < p.np; ++i) {
    if (!dropped && p.r[i] == 4) {
      dropped = true;
      continue;
    }
    rest[nr++] = p.r[i];
  }
  for (int i = 0; i < nr; ++i)
    for (int k = i + 1; k < nr; ++k)
      if (rest[k] > rest[i]) {
        const int t = rest[i];
        rest[i] = rest[k];
        rest[k] = t;
      }
  // a radix-2 last pass would leave N / 4 + 1 mirrored groups per transform (one transform per
  // work-group at n 600): where a radix 2 remains, it goes first among the middle passes and the
  // others follow in increasing order, so that the last pass has the largest radix
  bool has2 = false;
  for (int i = 0; i < nr; ++i) has2 = has2 || rest[i] == 2;
  if (!has2) {
    for (int i = 0; i < nr; ++i) q.r[q.np++] = rest[i];
  } else {
    for (int i = nr - 1; i >= 0; --i) q.r[q.np++] = rest[i];
  }
  return q;
}

template <int N>
struct Fp {
  static constexpr FftPlan plan = make_fused_plan(N);
  static constexpr int np = plan.np;
  static constexpr int R(int i) { return plan.r[i]; }
  static constexpr int Ns(int i) {
    int s = 1;
    for (int k = 0; k < i; ++k) s *= plan.r[k];
    return s;
  }
  static constexpr bool fusable = np >= 2 && plan.r[0] == 4 && N % 4 == 0;
};

// In-place Stockham pass P of F transforms held in LDS (transform f at buf + f N); each thread
// stages its butterflies' inputs in registers between two barriers.
template <int N, int F, int NT, int P>
__device__ __forceinline__ void lds_pass(float2* __restrict__ buf, const float2* __restrict__ tw2, int tid) {
  constexpr int R = Fp<N>::R(P);
  constexpr int Ns = Fp<N>::Ns(P);
  constexpr int nb = N / R;
  constexpr int TASKS = F * nb;
  constexpr int TPT = (TASKS + NT - 1) / NT;
  constexpr int tstep = N / (Ns * R);
  float2 v[TPT][R];
#pragma unroll
  for (int c = 0; c < TPT; ++c) {
    const int task = tid + c * NT;
    if (TASKS % NT == 0 || task < TASKS) {
      const int f = task / nb, j = task % nb;
#pragma unroll
      for (int t = 0; t < R; ++t) v[c][t] = buf[f * N + j + t * nb];
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < TPT; ++c) {
    const int task = tid + c * NT;
    if (TASKS % NT == 0 || task < TASKS) {
      const int f = task / nb, j = task % nb;
      const int jm = j % Ns;
      if constexpr (Ns > 1) {
#pragma unroll
        for (int t = 1; t < R; ++t)
          v[c][t] = cmul(v[c][t], tw2[2 * jm * t * tstep]);
      }
      Dft<R>::run(v[c]);
      const int base = (j / Ns) * Ns * R + jm;
#pragma unroll
      for (int t = 0; t < R; ++t) buf[f * N + base + t * Ns] = v[c][t];
    }
  }
  __syncthreads();
}

template <int N, int F, int NT, int P, int PEND>
__device__ __forceinline__ void lds_passes(float2* buf, const float2* tw2, int tid) {
  if constexpr (P < PEND) {
    lds_pass<N, F, NT, P>(buf, tw2, tid);
    lds_passes<N, F, NT, P + 1, PEND>(buf, tw2, tid);
  }
}

}  // namespace pfk
