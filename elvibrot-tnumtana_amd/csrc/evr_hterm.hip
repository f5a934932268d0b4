// FP64 H|psi> of one Smolyak term (sum-factorised), in register blocks.
//
// One workgroup applies one term to NV = 1 << lv vectors.  The term's basis
// tensor x lives in LDS as [function][vector]; the work runs in a few phases,
// each a pass over LDS with one barrier:
//
//  1. x is gathered and rotated, mode by mode, into the eigenvectors of the
//     mode's coordinate matrix Q = W x B (DVR; plans with a q-linear G only).
//     There Q is the diagonal xi, so G_ij(q) = c_ij + sum_k a_ijk q_k acts on
//     the modes k != i, j as a number per function.
//  2. V part: basis -> grid, V, grid -> basis (BDP_TO_GDP BGSG4:2385-2496,
//     GDP_TO_BDP BGSG4:2497-2581) over the modes with more than one function
//     (V summed over the others once per potential).  Neighbouring modes form
//     groups of one or two; a thread carries a group's block through its 1D
//     matrices in registers.  A step takes the fastest group of the LDS layout
//     and leaves it slowest, so its reads have the (odd) block stride and its
//     writes are consecutive; the last group goes up, through V and down
//     without leaving registers.
//  3. Kinetic part.  With P, T, U, R, S the basis-space factors of the slots
//     (W D1 B, W D1 D1 B, W D1 x D1 B, W D1 x B, W x D1 B; the reference's
//     grid form -1/2 sum_ij d_i G_ij(q) d_j, OPSG4:1548-1650, between
//     GDP_TO_BDP and BDP_TO_GDP) and g_ij = c_ij + sum_{k != i,j} a_ijk xi_k,
//       y += h x + sum_j [ g_jj T_j x + a_jjj U_j x ]
//              + sum_i P_i ( f_i x + sum_{j > i} (g_ij + g_ji) P_j x
//                                  + sum_{j != i} a_ijj (R_j + S_j) x ),
//     because operators of different modes commute and g_ij does not depend
//     on the functions of modes i and j.  A thread takes one pencil of NBP
//     functions of the term's pencil mode: it reads the pencils of the other
//     modes from LDS, forms every bracket M_i of its functions in registers
//     and writes them once; after one barrier the P_i are applied.
//  4. y is rotated back and written, weight applied, to the term's rows of R.
//
// What bounds it: latency.  A term is small (63 to 2,025 functions carry most
// of D=9 SG4 L=8) and a phase is one chain of LDS, scalar and FP64 latencies
// that workgroups hide from each other: the waves wait for 65% of their cycles,
// and 59% of the vector instructions are indices, addresses and moves of the 56
// registers that the kernel spills (17 kinetic variants and 16 block shapes
// share it).  So the phases are few (14 for a six-mode term, where applying one
// factor at a time between barriers took about 180), the kernel is held to 128
// VGPRs for 16 waves per CU, the coefficient rows are staged in LDS beside the
// factors, and a wave asks for the term's 1D matrices behind the gather, as
// they are read through the scalar cache (1% of its requests miss).  D=9 SG4
// L=8, 32 vectors, type 10 with q-linear G: 29.0 ms against 121.0 ms for the
// term kernels of evr_term.hip; D=6 L=5, 2 vectors 15.9 against 54.4 us; one
// vector at D=9 L=8 1.60 against 9.1 ms.
#include "evr_hblock.hpp"

namespace evr {

// Two modes of the last group, the one of fewer functions (second here) up,
// times V and down for every point of the other, whose matrices then stay in
// scalar registers over the loop when they are small.  Strides s1, s2 of the
// block's functions and v1, v2 of its points.
template <int B1, int N1, int B2, int N2, typename OUT>
__device__ __forceinline__ void top_pair(ctab pool, int mB1, int mB2, int mW1, int mW2, const double *__restrict__ vp,
                                         int blk, int v1, int v2, const double *in, int s1, int s2, OUT out)
{
  double t[B2][N1];
  {
    constexpr int C = hrows(N1, B1);
#pragma unroll
    for (int q0 = 0; q0 < N1; q0 += C) {
      const ctab M1 = pool + opaque(mB1);
#pragma unroll
      for (int b2 = 0; b2 < B2; ++b2) {
        double v[B1];
#pragma unroll
        for (int b = 0; b < B1; ++b) v[b] = in[b * s1 + b2 * s2];
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
  if constexpr (B2 * N2 <= 12) {
    const ctab MB = pool + opaque(mB2), MW = pool + opaque(mW2);
#pragma unroll
    for (int q1 = 0; q1 < N1; ++q1) {
      double u[N2];
#pragma unroll
      for (int q2 = 0; q2 < N2; ++q2) u[q2] = vp[(unsigned)(blk + v1 * q1 + v2 * q2)];
#pragma unroll
      for (int q2 = 0; q2 < N2; ++q2) {
        double a = MB[q2 * B2] * t[0][q1];
#pragma unroll
        for (int b = 1; b < B2; ++b) a = fma(MB[q2 * B2 + b], t[b][q1], a);
        u[q2] *= a;
      }
#pragma unroll
      for (int b = 0; b < B2; ++b) {
        double a = MW[b * N2] * u[0];
#pragma unroll
        for (int q2 = 1; q2 < N2; ++q2) a = fma(MW[b * N2 + q2], u[q2], a);
        t[b][q1] = a;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  } else {
#pragma unroll
    for (int q1 = 0; q1 < N1; ++q1) {
      double u[N2], w[B2];
#pragma unroll
      for (int q2 = 0; q2 < N2; ++q2) u[q2] = vp[(unsigned)(blk + v1 * q1 + v2 * q2)];
#pragma unroll
      for (int b = 0; b < B2; ++b) w[b] = t[b][q1];
      rows_apply<B2, N2>(pool, mB2, w, [&](int q2, double a) { u[q2] *= a; });
      rows_apply<N2, B2>(pool, mW2, u, [&](int b, double a) { t[b][q1] = a; });
    }
  }
#pragma unroll
  for (int b2 = 0; b2 < B2; ++b2)
    rows_apply<N1, B1>(pool, mW1, t[b2], [&](int b, double a) { out(b, b2, a); });
}

// the last group: up (B), times V (point q of block blk at vp[blk + vs q]),
// down (W)
template <int B1, int N1, int B2, int N2, typename OUT>
__device__ __forceinline__ void block_top(ctab pool, const HGroup EVR_CONST &G, const double *__restrict__ vp, int blk,
                                          int vs, const double *in, int s, OUT out)
{
  if constexpr (B2 == 1 && N2 == 1) {
    double t[1][N1];
    first_mode<B1, N1, 1>(pool, G.mB[0], in, s, t);
#pragma unroll
    for (int q = 0; q < N1; ++q) t[0][q] *= vp[(unsigned)(blk + vs * q)];
    __builtin_amdgcn_sched_barrier(0);
    rows_apply<N1, B1>(pool, G.mW[0], t[0], out);
  } else if constexpr (B1 < B2) {
    top_pair<B2, N2, B1, N1>(pool, G.mB[1], G.mB[0], G.mW[1], G.mW[0], vp, blk, vs * N1, vs, in, s * B1, s,
                             [&](int b2, int b1, double a) { out(b1 + B1 * b2, a); });
  } else {
    top_pair<B1, N1, B2, N2>(pool, G.mB[0], G.mB[1], G.mW[0], G.mW[1], vp, blk, vs, vs * N1, in, s, s * B1,
                             [&](int b1, int b2, double a) { out(b1 + B1 * b2, a); });
  }
}

// Rotation of a single mode of any extent nb (stride n1) from x to y, a thread
// per value: a block of one mode may be all there is, and one lane would then
// walk its nb x nb matrix alone (12 functions: 9 us a rotation).
__device__ __forceinline__ void rotate_generic(ctab M, int nb, int n1, int nunit, int lv, const double *x, double *y)
{
  const float rn1 = 1.0f / (float)n1, rnb = 1.0f / (float)nb;
  const int s = n1 << lv;
  for (int wk = threadIdx.x; wk < nunit; wk += blockDim.x) {
    const int r = fdiv(wk >> lv, n1, rn1), q = r - fdiv(r, nb, rnb) * nb;
    const double *in = x + (wk - q * s);
    const ctab row = M + q * nb;
    double a = row[0] * in[0];
    for (int b = 1; b < nb; ++b) a = fma(row[b], in[b * s], a);
    y[wk] = a;
  }
}

// generic last group (in and out may be the same)
template <typename OUT>
__device__ __forceinline__ void generic_top(ctab B, ctab W, int nb, int nq,
                                            const double *__restrict__ vp, int blk, int vs, const double *in, int s,
                                            OUT out)
{
  double r[kMaxNb];
#pragma unroll
  for (int i = 0; i < kMaxNb; ++i) r[i] = 0.0;
  for (int q = 0; q < nq; ++q) {
    double a = 0.0;
    for (int i = 0; i < nb; ++i) a = fma(B[q * nb + i], in[i * s], a);
    a *= vp[(unsigned)(blk + vs * q)];
#pragma unroll
    for (int i = 0; i < kMaxNb; ++i)
      if (i < nb) r[i] = fma(W[i * nq + q], a, r[i]);
  }
#pragma unroll
  for (int i = 0; i < kMaxNb; ++i)
    if (i < nb) out(i, r[i]);
}

template <int N, int K = 0, typename F>
__device__ __forceinline__ void unroll_for(F f)
{
  if constexpr (K < N) {
    f(std::integral_constant<int, K>{});
    unroll_for<N, K + 1>(f);
  }
}

// g = c + sum_k a_k xi_k of a coefficient row in LDS: NA values for the active
// modes, the constant, the value for the pencil mode; modes I, J and (with a
// pencil) 0 have no entry
template <int NBP, int NA, bool hasA, int I, int J>
__device__ __forceinline__ double hrow(const double *row, const double (&xi)[NA + 1])
{
  double g = row[NA];
  if constexpr (hasA) {
#pragma unroll
    for (int k = NBP > 1 ? 1 : 0; k < NA; ++k)
      if (k != I && k != J) g = fma(row[k], xi[k], g);
  }
  return g;
}

// Kinetic part of the term (phase 3 above) with NA active modes, added to y.
// sF: factors, then the coefficient rows; sx: x, sy: y, sm: nm arrays of M.
template <int NBP, int NA, int MODE>
__device__ __forceinline__ void keo_term(const HTerm EVR_CONST &term, const HArgs &a, const double *__restrict__ sF,
                                         const double *sx, double *sy, double *sm)
{
  const int nbt = term.nbt, lv = a.lv, NV = 1 << lv, tid = threadIdx.x;
  constexpr bool hasA = MODE == 2, hasM = MODE >= 1;
  const int stp = NBP > 1 ? term.st[0] : 1;
  const int nw = (nbt / NBP) << lv;
  const double *rows = sF + term.lC;
  constexpr int RL = hrow_len(NA);
  const double *alpha = rows + (1 + NA + NA * (NA - 1) / 2) * RL;  // [j NA + i]
  const double *fs = alpha + NA * NA;
  constexpr int I0 = NBP > 1 ? 1 : 0;  // M of the pencil mode stays in registers
  const float rstp = 1.0f / (float)stp;
  const int step = term.nm > 0 ? term.nm : 1;
  for (int i0 = I0; i0 == I0 || (hasM && i0 < NA); i0 += step) {
    for (int wk = tid; wk < nw; wk += blockDim.x) {
      const int v = wk & (NV - 1), r = wk >> lv;
      const int e0 = NBP > 1 ? r + fdiv(r, stp, rstp) * stp * (NBP - 1) : r;
      const HTerm EVR_CONST &td = (&term)[opaque(0)];
      double xi[NA + 1], xp[NBP], xr[NBP], y[NBP], M[NA + 1][NBP];
      int dig[NA + 1];
#pragma unroll
      for (int k = I0; k < NA; ++k) {
        const int st = td.st[k], nb = td.nb[k];
        const int q = fdiv(e0, st, td.rst[k]);
        dig[k] = q - fdiv(q, nb, td.rnb[k]) * nb;
        xi[k] = hasA ? sF[td.lF[k] + 4 * nb * nb + dig[k]] : 0.0;
      }
#pragma unroll
      for (int c = 0; c < NBP; ++c) {
        xp[c] = (NBP > 1 && hasA) ? sF[td.lF[0] + 4 * NBP * NBP + c] : 0.0;
        xr[c] = sx[((e0 + c * stp) << lv) + v];
      }
      {
        const double g = hrow<NBP, NA, hasA, -1, -1>(rows, xi);
        const double gp = NBP > 1 ? rows[NA + 1] : 0.0;
#pragma unroll
        for (int c = 0; c < NBP; ++c) {
          const double y0 = i0 == I0 ? sy[((e0 + c * stp) << lv) + v] : 0.0;
          y[c] = fma(fma(gp, xp[c], g), xr[c], y0);
        }
      }
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const double f = fs[i];
#pragma unroll
        for (int c = 0; c < NBP; ++c) M[i][c] = f * xr[c];
      }
      unroll_for<NA>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        __builtin_amdgcn_sched_barrier(0);
        double z[NBP], t[NBP], u[NBP], rs[NBP];
#pragma unroll
        for (int c = 0; c < NBP; ++c) z[c] = t[c] = u[c] = rs[c] = 0.0;
        const double *F = sF + td.lF[j];
        if constexpr (NBP > 1 && j == 0) {
#pragma unroll
          for (int c = 0; c < NBP; ++c)
#pragma unroll
            for (int b = 0; b < NBP; ++b) {
              const double *f = F + 4 * (c * NBP + b);
              z[c] = fma(f[0], xr[b], z[c]);
              t[c] = fma(f[1], xr[b], t[c]);
              u[c] = fma(f[2], xr[b], u[c]);
              rs[c] = fma(f[3], xr[b], rs[c]);
            }
        } else {
          const int st = td.st[j], nb = td.nb[j];
          const double *f = F + 4 * dig[j] * nb;
          const double *xs = sx + ((e0 - dig[j] * st) << lv) + v;
          auto one = [&](int b) {
            const double f0 = f[4 * b], f1 = f[4 * b + 1], f2 = f[4 * b + 2], f3 = f[4 * b + 3];
#pragma unroll
            for (int c = 0; c < NBP; ++c) {
              const double xv = xs[(b * st + c * stp) << lv];
              z[c] = fma(f0, xv, z[c]);
              t[c] = fma(f1, xv, t[c]);
              u[c] = fma(f2, xv, u[c]);
              rs[c] = fma(f3, xv, rs[c]);
            }
          };
          if (nb == 3) {
#pragma unroll
            for (int b = 0; b < 3; ++b) one(b);
          } else if (nb == 5) {
#pragma unroll
            for (int b = 0; b < 5; ++b) one(b);
          } else {
            for (int b = 0; b < nb; ++b) one(b);
          }
        }
        {
          const double *row = rows + (1 + j) * RL;
          const double g = hrow<NBP, NA, hasA, j, j>(row, xi);
          const double gp = NBP > 1 && j > 0 ? row[NA + 1] : 0.0;
#pragma unroll
          for (int c = 0; c < NBP; ++c) y[c] += fma(fma(gp, xp[c], g), t[c], u[c]);
        }
        if constexpr (hasM) {
          unroll_for<NA>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < j) {
              const double *row = rows + (1 + NA + j * (j - 1) / 2 + i) * RL;
              const double g = hrow<NBP, NA, hasA, i, j>(row, xi);
              const double gp = NBP > 1 && i > 0 ? row[NA + 1] : 0.0;
#pragma unroll
              for (int c = 0; c < NBP; ++c) M[i][c] = fma(fma(gp, xp[c], g), z[c], M[i][c]);
            }
            if constexpr (i != j) {
              if constexpr (hasA) {
                const double al = alpha[j * NA + i];
#pragma unroll
                for (int c = 0; c < NBP; ++c) M[i][c] = fma(al, rs[c], M[i][c]);
              }
            }
          });
        }
        // the brackets are complete for mode j here: left to itself the compiler
        // keeps every mode's inputs alive to the end and spills
#pragma unroll
        for (int c = 0; c < NBP; ++c) {
          pin(y[c]);
#pragma unroll
          for (int i = 0; i < NA; ++i) pin(M[i][c]);
        }
      });
      if (i0 == I0) {
        if (NBP > 1 && hasM) {
          const double *F = sF + td.lF[0];
#pragma unroll
          for (int c = 0; c < NBP; ++c)
#pragma unroll
            for (int b = 0; b < NBP; ++b) y[c] = fma(F[4 * (c * NBP + b)], M[0][b], y[c]);
        }
#pragma unroll
        for (int c = 0; c < NBP; ++c) sy[((e0 + c * stp) << lv) + v] = y[c];
      }
      if (hasM) {
#pragma unroll
        for (int i = I0; i < NA; ++i)
          if (i >= i0 && i < i0 + step) {
            double *o = sm + (((i - i0) * nbt) << lv);
#pragma unroll
            for (int c = 0; c < NBP; ++c) o[((e0 + c * stp) << lv) + v] = M[i][c];
          }
      }
    }
    if (!hasM || NA <= I0) break;
    __syncthreads();
    const int i1 = NA < i0 + step ? NA : i0 + step;
    for (int wk = tid; wk < nw; wk += blockDim.x) {
      const int v = wk & (NV - 1), r = wk >> lv;
      const int e0 = NBP > 1 ? r + fdiv(r, stp, rstp) * stp * (NBP - 1) : r;
      const HTerm EVR_CONST &td = (&term)[opaque(0)];
      double y[NBP];
#pragma unroll
      for (int c = 0; c < NBP; ++c) y[c] = sy[((e0 + c * stp) << lv) + v];
      for (int i = i0; i < i1; ++i) {
        const int st = td.st[i], nb = td.nb[i];
        const int q = fdiv(e0, st, td.rst[i]);
        const int n = q - fdiv(q, nb, td.rnb[i]) * nb;
        const double *f = sF + td.lF[i] + 4 * n * nb;
        const double *ms = sm + (((i - i0) * nbt + e0 - n * st) << lv) + v;
        auto one = [&](int b) {
          const double f0 = f[4 * b];
#pragma unroll
          for (int c = 0; c < NBP; ++c) y[c] = fma(f0, ms[(b * st + c * stp) << lv], y[c]);
        };
        if (nb == 3) {
#pragma unroll
          for (int b = 0; b < 3; ++b) one(b);
        } else if (nb == 5) {
#pragma unroll
          for (int b = 0; b < 5; ++b) one(b);
        } else {
          for (int b = 0; b < nb; ++b) one(b);
        }
      }
#pragma unroll
      for (int c = 0; c < NBP; ++c) sy[((e0 + c * stp) << lv) + v] = y[c];
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(1024, 4) void k_hterm(HArgs a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *sF = reinterpret_cast<double *>(smem_raw);
  const int lv = a.lv, NV = 1 << lv, tid = threadIdx.x, nt = blockDim.x;
  // all vector tiles of a term on one XCD (workgroups go round-robin over the
  // 8), the cost-sorted terms dealt to the XCDs in turn
  const int nvt = (a.nvec + NV - 1) >> lv;
  const int b = (int)blockIdx.x;
  const int slot = b >> 3, vt = slot % nvt;
  const int t = a.order[(slot / nvt) * 8 + (b & 7)];
  if (t < 0) return;
  const HTerm EVR_CONST &td = a.terms[t];
  const int v0 = vt << lv, nbt = td.nbt, nunit = nbt << lv, ng = td.ng;
  double *sx = sF + td.fw, *sy = sx + nunit, *sw = sy + nunit;
  const HGroup EVR_CONST *G = a.groups + td.g0;

  // Every phase below reads the term's 1D matrices at uniform addresses, and a
  // miss costs a phase about a thousand cycles of one serial chain; the last
  // wave asks for all of them at once, behind the gather.
  if (__builtin_amdgcn_readfirstlane(tid >> 6) == (nt >> 6) - 1) {
    touch((ctab)&td, sizeof(HTerm) / 8);
    touch((ctab)G, ng * (int)(sizeof(HGroup) / 8));
    for (int g = 0; g < ng; ++g) {
      touch(a.pool + G[g].mB[0], G[g].pw[0]);
      if (G[g].pw[1] > 0) touch(a.pool + G[g].mB[1], G[g].pw[1]);
    }
  }

  // the active modes' factors and the coefficient rows, one flat pass
  if (a.hasKeo) {
    const int na = td.na, lC = td.lC, fw = td.fw;
    for (int i = tid; i < fw; i += nt) {
      int base = 0, src = na ? td.gF[0] : 0;
      for (int m = 1; m < na; ++m)
        if (td.lF[m] <= i) {
          base = td.lF[m];
          src = td.gF[m];
        }
      sF[i] = i >= lC ? a.coef[td.coef + (i - lC)] : a.fpool[src + (i - base)];
    }
  }
  // x, the first group rotated on the way in; groups of any shape rotate from
  // one of the two tensors to the other, the last of them into sx
  {
    double *px = a.hasA && (td.ngen & 1) ? sy : sx, *py = a.hasA && (td.ngen & 1) ? sx : sy;
    const int *mp = a.map + td.off_nb;
    const bool rot = a.hasA && ng > 0 && G[0].kind != kHgGeneric;
    if (rot) {
      const int nb = G[0].nb, nblk = nbt / nb;
      for (int wk = tid; wk < nblk << lv; wk += nt) {
        const int v = wk & (NV - 1), blk = wk >> lv;
        const int col = v0 + v < a.nvec ? v0 + v : a.nvec - 1;
        const int *m = mp + blk * nb;
        double *o = px + ((blk * nb) << lv) + v;
        const int sv = opaque(NV);
        double in[25];
        switch (G[0].kind > kHgSquare ? G[0].kind : G[0].kind + kHgSquare) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K: {                                                                                          \
    _Pragma("unroll") for (int i = 0; i < B1 * B2; ++i)                                              \
    {                                                                                                \
      const int pk = m[i];                                                                           \
      const double xv = X_AT(pk);                                                                    \
      in[i] = pk >= 0 ? xv : 0.0;                                                                    \
    }                                                                                                \
    block_apply<B1, N1, B2, N2>(a.pool, G[0].mI[0], G[0].mI[1], in, 1,                               \
                                [&](int i, double val) { o[i * sv] = val; });                        \
    break;                                                                                           \
  }
#define X_AT(pk) a.X[(int64_t)((pk) >= 0 ? (pk) : 0) * a.nvec + col]
          EVR_HG_SQUARE(X)
#undef X
          default: break;
        }
      }
    } else {
      for (int wk = tid; wk < nunit; wk += nt) {
        const int v = wk & (NV - 1), e = wk >> lv;
        const int col = v0 + v < a.nvec ? v0 + v : a.nvec - 1;
        const int pk = mp[e];
        const double xv = X_AT(pk);
        px[wk] = pk >= 0 ? xv : 0.0;
      }
    }
#undef X_AT
    __syncthreads();
    if (a.hasA) {
      for (int g = rot ? 1 : 0; g < ng; ++g) {
        const int nb = G[g].nb, n1 = G[g].n1, nblk = nbt / nb;
        if (G[g].kind == kHgGeneric) {
          rotate_generic(a.pool + G[g].mI[0], nb, n1, nunit, lv, px, py);
          double *const t = px;
          px = py;
          py = t;
          __syncthreads();
          continue;
        }
        const float rn1 = 1.0f / (float)n1;
        for (int wk = tid; wk < nblk << lv; wk += nt) {
          const int v = wk & (NV - 1), blk = wk >> lv;
          const int i3 = fdiv(blk, n1, rn1);
          double *io = px + ((blk + i3 * n1 * (nb - 1)) << lv) + v;
          const int s = opaque(n1 << lv);
          switch (G[g].kind > kHgSquare ? G[g].kind : G[g].kind + kHgSquare) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K: {                                                                                          \
    double o_[B1 * B2];                                                                              \
    block_apply<B1, N1, B2, N2>(a.pool, G[g].mI[0], G[g].mI[1], io, s,                               \
                                [&](int i, double val) { o_[i] = val; });                            \
    _Pragma("unroll") for (int i = 0; i < B1 * B2; ++i) io[i * s] = o_[i];                           \
    break;                                                                                           \
  }
            EVR_HG_SQUARE(X)
#undef X
            default: break;
          }
        }
        __syncthreads();
      }
    }
  }

  // V part, written to y (a slabbed one is summed there)
  if (!a.hasV || td.QO > 1) {
    for (int wk = tid; wk < nunit; wk += nt) sy[wk] = 0.0;
    __syncthreads();
  }
  if (a.hasV) {
    const double *Vt = a.V + td.off_vq;
    if (ng == 0) {
      for (int v = tid; v < NV; v += nt) sy[v] = Vt[0] * sx[v];
      __syncthreads();
    } else {
      double *bufA = sw, *bufB = sw + (td.wA << lv), *xs = bufB + (td.wB << lv), *cr = xs + (td.nbI << lv);
      const int QO = td.QO, nbO = td.nbO, nbI = td.nbI;
      int64_t qin = 1;  // points of the inner modes
      for (int g = 0; g < ng - td.nO; ++g) qin *= G[g].nq;
      const int gi = ng - td.nO;  // inner groups
      for (int qO = 0; qO < QO; ++qO) {
        const double *src = sx;
        if (QO > 1) {
          // Kronecker rows of the outer modes at this outer point
          for (int bo = tid; bo < nbO; bo += nt) {
            int rb = bo, rq = qO;
            double cb = 1.0, cw = 1.0;
            for (int d = 0; d < td.nOm; ++d) {
              const int nb = td.onb[d], nq = td.onq[d];
              const int bb = rb % nb, qq = rq % nq;
              rb /= nb;
              rq /= nq;
              cb *= a.pool[td.oB[d] + qq * nb + bb];
              cw *= a.pool[td.oW[d] + bb * nq + qq];
            }
            cr[bo] = cb;
            cr[nbO + bo] = cw;
          }
          __syncthreads();
          for (int wk = tid; wk < nbI << lv; wk += nt) {
            double s = 0.0;
            for (int bo = 0; bo < nbO; ++bo) s = fma(cr[bo], sx[wk + ((bo * nbI) << lv)], s);
            xs[wk] = s;
          }
          __syncthreads();
          src = xs;
        }
        const double *Vq = Vt + qin * qO;
        // up: group g fastest in, slowest out
        int cur = nbI;
        double *dst = bufA;
        for (int g = 0; g + 1 < gi; ++g) {
          const int nb = G[g].nb, nblk = cur / nb;
          for (int wk = tid; wk < nblk << lv; wk += nt) {
            const int v = wk & (NV - 1), blk = wk >> lv;
            const double *in = src + ((blk * nb) << lv) + v;
            double *o = dst + wk;
            const int sv = opaque(NV), so = opaque(nblk << lv);
            switch (G[g].kind) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K:                                                                                            \
    block_apply<B1, N1, B2, N2>(a.pool, G[g].mB[0], G[g].mB[1], in, sv,                              \
                                [&](int i, double val) { o[i * so] = val; });                        \
    break;
              EVR_HG_KINDS(X)
#undef X
              default:
                block_generic(a.pool + G[g].mB[0], nb, G[g].nq, in, sv, [&](int i, double val) { o[i * so] = val; });
            }
          }
          __syncthreads();
          cur = nblk * G[g].nq;
          src = dst;
          dst = dst == bufA ? bufB : bufA;
        }
        // last inner group: up, V, down; in place except from x itself
        {
          const int g = gi - 1, nb = G[g].nb, nblk = cur / nb;
          double *out = gi == 1 ? (QO == 1 ? sy : xs) : const_cast<double *>(src);
          for (int wk = tid; wk < nblk << lv; wk += nt) {
            const int v = wk & (NV - 1), blk = wk >> lv;
            const double *in = src + ((blk * nb) << lv) + v;
            double *o = out + ((blk * nb) << lv) + v;
            const int sv = opaque(NV), ns = opaque(nblk);
            switch (G[g].kind) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K:                                                                                            \
    block_top<B1, N1, B2, N2>(a.pool, G[g], Vq, blk, ns, in, sv,                                     \
                              [&](int i, double val) { o[i * sv] = val; });                          \
    break;
              EVR_HG_KINDS(X)
#undef X
              default:
                generic_top(a.pool + G[g].mB[0], a.pool + G[g].mW[0], nb, G[g].nq, Vq, blk, ns, in, sv,
                            [&](int i, double val) { o[i * sv] = val; });
            }
          }
          __syncthreads();
          src = out;
        }
        // down: group g slowest in, fastest out; the first group ends in y
        for (int g = gi - 2; g >= 0; --g) {
          const int nb = G[g].nb, nq = G[g].nq, nblk = cur / nq;
          double *out = g == 0 ? (QO == 1 ? sy : xs) : dst;
          for (int wk = tid; wk < nblk << lv; wk += nt) {
            const int v = wk & (NV - 1), blk = wk >> lv;
            const double *in = src + wk;
            double *o = out + ((blk * nb) << lv) + v;
            const int sv = opaque(NV), si = opaque(nblk << lv);
            switch (G[g].kind) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K:                                                                                            \
    block_apply<N1, B1, N2, B2>(a.pool, G[g].mW[0], G[g].mW[1], in, si,                              \
                                [&](int i, double val) { o[i * sv] = val; });                        \
    break;
              EVR_HG_KINDS(X)
#undef X
              default:
                block_generic(a.pool + G[g].mW[0], nq, nb, in, si, [&](int i, double val) { o[i * sv] = val; });
            }
          }
          __syncthreads();
          cur = nblk * nb;
          src = out;
          dst = dst == bufA ? bufB : bufA;
        }
        if (QO > 1) {
          for (int wk = tid; wk < nunit; wk += nt) {
            const int e = wk >> lv, v = wk & (NV - 1);
            const int bo = e / nbI;
            sy[wk] = fma(cr[nbO + bo], xs[((e - bo * nbI) << lv) + v], sy[wk]);
          }
          __syncthreads();
        }
      }
    }
  }

  // kinetic part, added to y
  if (a.hasKeo) {
    __syncthreads();
    auto keo = [&](auto mode) {
      constexpr int MODE = decltype(mode)::value;
#define X(NBP, NA)                                                                                   \
  case NA: keo_term<NBP, NA, MODE>(td, a, sF, sx, sy, sw); break;
      if (td.nbp == 3) {
        switch (td.na) {
          X(3, 1) X(3, 2) X(3, 3) X(3, 4) X(3, 5) X(3, 6) X(3, 7) X(3, 8)
          default: break;
        }
      } else {
        switch (td.na) {
          X(1, 0) X(1, 1) X(1, 2) X(1, 3) X(1, 4) X(1, 5) X(1, 6) X(1, 7) X(1, 8)
          default: break;
        }
      }
#undef X
    };
    if (a.hasA) keo(std::integral_constant<int, 2>{});
    else if (a.hasM) keo(std::integral_constant<int, 1>{});
    else keo(std::integral_constant<int, 0>{});
  }
  __syncthreads();

  // rotate back and write the term rows
  {
    const int *rp = a.rowpos + td.off_nb;
    const double w = td.w;
    double *px = sx, *py = sy;
    if (a.hasA) {
      for (int g = 0; g < ng; ++g) {
        const int nb = G[g].nb, n1 = G[g].n1, nblk = nbt / nb;
        if (G[g].kind == kHgGeneric) {
          rotate_generic(a.pool + G[g].mO[0], nb, n1, nunit, lv, py, px);
          double *const t = px;
          px = py;
          py = t;
          __syncthreads();
          continue;
        }
        const float rn1 = 1.0f / (float)n1;
        for (int wk = tid; wk < nblk << lv; wk += nt) {
          const int v = wk & (NV - 1), blk = wk >> lv;
          const int i3 = fdiv(blk, n1, rn1);
          double *io = py + ((blk + i3 * n1 * (nb - 1)) << lv) + v;
          const int s = opaque(n1 << lv);
          switch (G[g].kind > kHgSquare ? G[g].kind : G[g].kind + kHgSquare) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K: {                                                                                          \
    double o_[B1 * B2];                                                                              \
    block_apply<B1, N1, B2, N2>(a.pool, G[g].mO[0], G[g].mO[1], io, s,                               \
                                [&](int i, double val) { o_[i] = val; });                            \
    _Pragma("unroll") for (int i = 0; i < B1 * B2; ++i) io[i * s] = o_[i];                           \
    break;                                                                                           \
  }
            EVR_HG_SQUARE(X)
#undef X
            default: break;
          }
        }
        __syncthreads();
      }
    }
    for (int wk = tid; wk < nunit; wk += nt) {
      const int v = wk & (NV - 1), e = wk >> lv;
      const int row = rp[e];
      if (row >= 0 && v0 + v < a.nvec) a.R[(int64_t)row * a.nvec + v0 + v] = w * py[wk];
    }
  }
}

hipError_t launch_hterm(const HArgs &a, int64_t nblk, int nt, size_t lds, hipStream_t s)
{
  // the dispatch grid is counted in work-items in 32 bits
  if (nblk > (int64_t)0xFFFFFFFFu / nt) return hipErrorInvalidConfiguration;
  (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_hterm), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds);
  hipLaunchKernelGGL(k_hterm, dim3((unsigned)nblk), dim3(nt), lds, s, a);
  return hipGetLastError();
}

}  // namespace evr
