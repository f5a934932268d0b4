// Basis <-> grid transforms of the Smolyak terms (BDP_TO_GDP BGSG4:2385-2496,
// GDP_TO_BDP BGSG4:2497-2581 with the weighted scatter BGSG4:951-1028).
//
// One workgroup takes one term and one vector.  The modes with more than one
// function go through the register blocks of evr_hblock.hpp in LDS; the
// one-function modes, whose B is a column and W a row, are expanded on the way
// out and contracted on the way in.  Consecutive threads take consecutive
// points of the full term grid in both directions, whatever modes they belong
// to: the grid point p = pl + Pl ph is split into a low part of 128 points or
// more and the rest, and two tables per part (the part's share of the reduced
// point, the product of its one-function entries) replace the digits.
//
// Bound: HBM, the grid vector is written or read once.  D=12 SG4 L=4, one
// vector out (84e6 points, 0.67 GB): 0.158 ms, 4.2 TB/s, against 9.89 ms for the
// one workgroup per term of the term kernel, which walked the outer points of
// every term and all combinations of its one-function modes serially.  D=9 SG4
// L=6, four vectors back (276e6 points, 2.2 GB): 0.65 ms, 3.4 TB/s, against 2.83
// ms.  A low part of 64 points measured slower (0.218 and 0.665 ms), four r
// points per wave too (0.73 ms: more LDS, fewer workgroups).  Small grids run in
// workgroups of one wave.
#include "evr_hblock.hpp"

namespace evr {

// Point i of the modes d0 .. d1-1 of a term: its r part, its number c among the
// one-function combinations, and their product (B, or W with w1).
__device__ __forceinline__ void xpart(const XTerm EVR_CONST &td, const double *__restrict__ pool1, int d0, int d1,
                                      int i, bool w1, int &r, int &c, double &s)
{
  int rs = 1, cs = 1;
  r = c = 0;
  s = 1.0;
  for (int d = d0; d < d1; ++d) {
    const int nq = td.nq[d], o = td.one[d];
    const int n = fdiv(i, nq, 1.0f / (float)nq), q = i - n * nq;
    i = n;
    if (o >= 0) {
      s *= pool1[o + (w1 ? nq : 0) + q];
      c += cs * q;
      cs *= nq;
    } else {
      r += rs * q;
      rs *= nq;
    }
  }
}

__global__ __launch_bounds__(kXThreads, 4) void k_b2g(XArgs a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int v = (int)(blockIdx.x % (unsigned)a.nvec);
  const XTerm EVR_CONST &td = a.terms[a.order[blockIdx.x / (unsigned)a.nvec]];
  const HGroup EVR_CONST *G = a.groups + td.g0;
  const int nbt = td.nbt, ng = td.ng, Pl = td.Pl, Ph = td.Ph, Rl = td.Rl;
  double *sx = reinterpret_cast<double *>(smem_raw), *bufA = sx + nbt, *bufB = bufA + td.wA;
  double *sl = bufB + td.wB, *sh = sl + Pl;  // one-function products
  int *rl = reinterpret_cast<int *>(sh + Ph), *rh = rl + Pl;
  for (int e = tid; e < nbt; e += nt) {
    const int pk = a.map[td.off_nb + e];
    sx[e] = pk >= 0 ? a.X[(int64_t)pk * a.nvec + v] : 0.0;
  }
  for (int i = tid; i < Pl + Ph; i += nt) {
    const bool hi = i >= Pl;
    int r, c;
    double s;
    xpart(td, a.pool1, hi ? td.nlow : 0, hi ? td.D : td.nlow, hi ? i - Pl : i, false, r, c, s);
    sl[i] = s;
    rl[i] = hi ? r * Rl : r;
  }
  __syncthreads();
  const double *src = sx;
  double *dst = bufA;
  int cur = nbt;
  for (int g = 0; g < ng; ++g) {
    const int nb = G[g].nb, nblk = cur / nb;
    for (int blk = tid; blk < nblk; blk += nt) {
      const double *in = src + blk * nb;
      double *o = dst + blk;
      const int so = opaque(nblk);
      switch (G[g].kind) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K:                                                                                            \
    block_apply<B1, N1, B2, N2>(a.pool, G[g].mP[0], G[g].mP[1], in, 1,                               \
                                [&](int i, double val) { o[i * so] = val; });                        \
    break;
        EVR_HG_KINDS(X)
#undef X
        default:
          block_generic(a.pool + G[g].mP[0], nb, G[g].nq, in, 1, [&](int i, double val) { o[i * so] = val; });
      }
    }
    __syncthreads();
    cur = nblk * G[g].nq;
    src = dst;
    dst = dst == bufA ? bufB : bufA;
  }
  double *out = a.G + (int64_t)v * a.gld + td.off_nq;
  const float rPl = 1.0f / (float)Pl;
  const int nqt = td.nqt;
  for (int p = tid; p < nqt; p += nt) {
    const int ph = fdiv(p, Pl, rPl), pl = p - ph * Pl;
    out[p] = src[rl[pl] + rh[ph]] * (sl[pl] * sh[ph]);
  }
}

// Contraction of the one-function modes on the way in: a wave takes N r points
// of the high part at a time (one where there are few), sums the high
// combinations in registers and the low ones through its own words of LDS.
template <int N>
__device__ __forceinline__ void g2b_rows(const double *__restrict__ in, int Pl, int Rl, int Cl, int Rh, int Ch,
                                         const int *pr, const int *pc, const int *plr, const int *plc,
                                         const double *sc, const double *sl, double *red, double *buf)
{
  const int nt = blockDim.x, nl = nt < 64 ? nt : 64, lane = threadIdx.x % nl, wave = threadIdx.x / nl, nw = nt / nl;
  double *tmp = buf + wave * kXRows * Pl;
  const float rRl = 1.0f / (float)Rl;
  for (int h0 = wave * N; h0 < Rh; h0 += nw * N) {
    int ho[N];  // first points, the last row again past the end
#pragma unroll
    for (int k = 0; k < N; ++k) ho[k] = Pl * pr[h0 + k < Rh ? h0 + k : Rh - 1];
    for (int pl = lane; pl < Pl; pl += 2 * nl) {
      const bool two = pl + nl < Pl;
      const double *q = in + pl;
      const int o2 = two ? nl : 0;
      double s0[N], s1[N];
#pragma unroll
      for (int k = 0; k < N; ++k) s0[k] = s1[k] = 0.0;
#pragma unroll 4
      for (int c = 0; c < Ch; ++c) {
        const int o = Pl * pc[c];
        const double w = sc[c];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          s0[k] = fma(w, q[o + ho[k]], s0[k]);
          s1[k] = fma(w, q[o + ho[k] + o2], s1[k]);
        }
      }
      const double w0 = sl[pl], w1 = sl[pl + o2];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        if (h0 + k >= Rh) break;
        double *o = Cl == 1 ? red + (h0 + k) * Rl : tmp + k * Pl;  // Pl = Rl with Cl = 1
        o[pl] = s0[k] * w0;
        if (two) o[pl + nl] = s1[k] * w1;
      }
    }
    if (Cl == 1) continue;
    // the wave's own words: LDS keeps a wave's order, the compiler is held to it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int nr = (h0 + N <= Rh ? N : Rh - h0) * Rl;
    for (int i = lane; i < nr; i += nl) {
      const int k = fdiv(i, Rl, rRl), r = i - k * Rl;
      const double *q = tmp + k * Pl + plr[r];
      double s = 0.0;
#pragma unroll 4
      for (int c = 0; c < Cl; ++c) s += q[plc[c]];
      red[h0 * Rl + i] = s;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

__global__ __launch_bounds__(kXThreads, 4) void k_g2b(XArgs a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int v = (int)(blockIdx.x % (unsigned)a.nvec);
  const XTerm EVR_CONST &td = a.terms[a.order[blockIdx.x / (unsigned)a.nvec]];
  const HGroup EVR_CONST *G = a.groups + td.g0;
  const int ng = td.ng, Pl = td.Pl, Ph = td.Ph, Rl = td.Rl, Rh = td.Rh;
  const int Cl = Pl / Rl, Ch = Ph / Rh;
  double *bufA = reinterpret_cast<double *>(smem_raw), *bufB = bufA + td.uA;  // bufA: the reduced grid
  double *sl = bufB + td.uB, *sc = sl + Pl;   // W products: of the low points, of the high combinations
  int *pc = reinterpret_cast<int *>(sc + Ch), *pr = pc + Ch;        // high combinations and r points: their ph
  int *plc = pr + Rh, *plr = plc + Cl;                              // the same of the low part: their pl
  for (int i = tid; i < Pl + Ph; i += nt) {
    const bool hi = i >= Pl;
    int r, c;
    double s;
    xpart(td, a.pool1, hi ? td.nlow : 0, hi ? td.D : td.nlow, hi ? i - Pl : i, true, r, c, s);
    if (hi) {
      if (r == 0) {
        pc[c] = i - Pl;
        sc[c] = s;
      }
      if (c == 0) pr[r] = i - Pl;
    } else {
      sl[i] = s;
      if (r == 0) plc[c] = i;
      if (c == 0) plr[r] = i;
    }
  }
  __syncthreads();
  // contract the one-function modes
  {
    const double *in = a.Gin + (int64_t)v * a.gld + td.off_nq;
    const int nw = nt < 64 ? 1 : nt >> 6;  // waves
    if (Rh >= kXRows * nw) g2b_rows<kXRows>(in, Pl, Rl, Cl, Rh, Ch, pr, pc, plr, plc, sc, sl, bufA, bufB);
    else g2b_rows<1>(in, Pl, Rl, Cl, Rh, Ch, pr, pc, plr, plc, sc, sl, bufA, bufB);
  }
  __syncthreads();
  const double *src = bufA;
  double *dst = bufB;
  int cur = td.nvq;
  for (int g = ng - 1; g >= 0; --g) {
    const int nb = G[g].nb, nq = G[g].nq, nblk = cur / nq;
    for (int blk = tid; blk < nblk; blk += nt) {
      const double *ip = src + blk;
      double *o = dst + blk * nb;
      const int si = opaque(nblk);
      switch (G[g].kind) {
#define X(K, B1, N1, B2, N2)                                                                         \
  case K:                                                                                            \
    block_apply<N1, B1, N2, B2>(a.pool, G[g].mQ[0], G[g].mQ[1], ip, si,                              \
                                [&](int i, double val) { o[i] = val; });                             \
    break;
        EVR_HG_KINDS(X)
#undef X
        default:
          block_generic(a.pool + G[g].mQ[0], nq, nb, ip, si, [&](int i, double val) { o[i] = val; });
      }
    }
    __syncthreads();
    cur = nblk * nb;
    src = dst;
    dst = dst == bufA ? bufB : bufA;
  }
  const double w = td.w;
  for (int e = tid; e < td.nbt; e += nt) {
    const int row = a.rowpos[td.off_nb + e];
    if (row >= 0) a.R[(int64_t)row * a.nvec + v] = w * src[e];
  }
}

size_t xform_words(const XTerm &t, bool b2g)
{
  const size_t tables = (size_t)t.Pl + t.Ph + (t.Pl + t.Ph + 1) / 2;
  if (b2g) return (size_t)t.nbt + t.wA + t.wB + tables;
  const size_t Cl = t.Pl / t.Rl, Ch = t.Ph / t.Rh;
  return (size_t)t.uA + t.uB + t.Pl + Ch + (Ch + t.Rh + Cl + t.Rl + 1) / 2;
}

hipError_t launch_xform(const XArgs &a, bool b2g, int64_t nterms, int nt, size_t lds, hipStream_t s)
{
  const int64_t nblk = nterms * a.nvec;
  if (nblk <= 0) return hipSuccess;
  // the dispatch grid is counted in work-items in 32 bits
  if (nblk > (int64_t)0xFFFFFFFFu / nt) return hipErrorInvalidConfiguration;
  if (b2g) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_b2g), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
    hipLaunchKernelGGL(k_b2g, dim3((unsigned)nblk), dim3(nt), lds, s, a);
  } else {
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_g2b), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
    hipLaunchKernelGGL(k_g2b, dim3((unsigned)nblk), dim3(nt), lds, s, a);
  }
  return hipGetLastError();
}

}  // namespace evr
