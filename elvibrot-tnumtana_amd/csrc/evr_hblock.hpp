// Register-block contractions shared by the H|psi> and transform kernels.
#pragma once
#include "evr_hterm.hpp"

namespace evr {

// A uniform value whose loads and multiples stay inside the loop that uses
// them: hoisted (1D matrices of two modes, the strides of a block, the
// extents of every mode) they exceed the scalar registers.
__device__ __forceinline__ int opaque(int p)
{
  asm volatile("" : "+s"(p));
  return p;
}

// the value is formed here, neither earlier nor later
__device__ __forceinline__ void pin(double &v)
{
  asm volatile("" : "+v"(v));
}

// Reads one word of every 64-byte line of n words at p, eight loads in flight:
// brings a term's tables into the scalar cache.
__device__ __forceinline__ void touch(ctab p, int n)
{
  const int EVR_CONST *q = (const int EVR_CONST *)p;
  const int last = 2 * n - 1;
  int sum = 0;
  for (int i = 0; i <= last; i += 8 * 16) {
    int w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = q[i + 16 * k < last ? i + 16 * k : last];
#pragma unroll
    for (int k = 0; k < 8; ++k) sum += w[k];
  }
  asm volatile("" ::"s"(sum));
}

// rows of an N x B matrix taken at a time: their coefficients have to fit the
// scalar registers beside the kernel's own values (32 words at most; 16 halves
// the waits' length but doubles their number: 34.0 against 32.3 ms at D=9 L=8,
// 52.8 against 54.3 us at D=6 L=5)
constexpr int hrows(int n, int b) { return n * b <= 32 ? n : (b >= 32 ? 1 : 32 / b); }

// out(o, value) for the N x B matrix at pool + m applied to v
template <int B, int N, typename OUT>
__device__ __forceinline__ void rows_apply(ctab pool, int m, const double (&v)[B], OUT out)
{
  constexpr int C = hrows(N, B);
#pragma unroll
  for (int q0 = 0; q0 < N; q0 += C) {
    const ctab M = pool + opaque(m);
#pragma unroll
    for (int q = q0; q < q0 + C && q < N; ++q) {
      double a = M[q * B] * v[0];
#pragma unroll
      for (int b = 1; b < B; ++b) a = fma(M[q * B + b], v[b], a);
      out(q, a);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// t[b2][q1] = sum_b1 M1(q1, b1) in(b1, b2); M1 N1 x B1 (the
// inputs are read again for every chunk of its rows)
template <int B1, int N1, int B2>
__device__ __forceinline__ void first_mode(ctab pool, int m1, const double *in, int s, double (&t)[B2][N1])
{
  constexpr int C = hrows(N1, B1);
#pragma unroll
  for (int q0 = 0; q0 < N1; q0 += C) {
    const ctab M1 = pool + opaque(m1);
#pragma unroll
    for (int b2 = 0; b2 < B2; ++b2) {
      double v[B1];
#pragma unroll
      for (int b = 0; b < B1; ++b) v[b] = in[(b + B1 * b2) * s];
#pragma unroll
      for (int q = q0; q < q0 + C && q < N1; ++q) {
        double a = M1[q * B1] * v[0];
#pragma unroll
        for (int b = 1; b < B1; ++b) a = fma(M1[q * B1 + b], v[b], a);
        t[b2][q] = a;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// out(q + N j, value): the N x B matrix at pool + m applied to the rows
// t[.][j] of a block
template <int B, int N, int J, typename OUT>
__device__ __forceinline__ void second_mode(ctab pool, int m, const double (&t)[B][J], OUT out)
{
  constexpr int C = hrows(N, B);
#pragma unroll
  for (int q0 = 0; q0 < N; q0 += C) {
    const ctab M = pool + opaque(m);
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int q = q0; q < q0 + C && q < N; ++q) {
        double a = M[q * B] * t[0][j];
#pragma unroll
        for (int b = 1; b < B; ++b) a = fma(M[q * B + b], t[b][j], a);
        out(j, q, a);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// the block (B1 x B2) at `in` (element stride s) through M1 (N1 x B1) and M2
// (N2 x B2): out(q1 + N1 q2, value)
template <int B1, int N1, int B2, int N2, typename OUT>
__device__ __forceinline__ void block_apply(ctab pool, int m1, int m2, const double *in, int s,
                                            OUT out)
{
  double t[B2][N1];
  first_mode<B1, N1, B2>(pool, m1, in, s, t);
  if constexpr (B2 == 1 && N2 == 1) {
#pragma unroll
    for (int q = 0; q < N1; ++q) out(q, t[0][q]);
  } else {
    second_mode<B2, N2, N1>(pool, m2, t, [&](int q1, int q2, double a) { out(q1 + N1 * q2, a); });
  }
}

// generic single mode: out(q) = sum_b M(q, b) in(b), the inputs read per result
template <typename OUT>
__device__ __forceinline__ void block_generic(ctab M, int nin, int nout, const double *in,
                                              int s, OUT out)
{
  for (int q = 0; q < nout; ++q) {
    double a = 0.0;
    for (int b = 0; b < nin; ++b) a = fma(M[q * nin + b], in[b * s], a);
    out(q, a);
  }
}

}  // namespace evr
