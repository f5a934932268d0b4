// The reference's grid form of one term with G, J, s per grid point
// (OPSG4:1566-1632), from psi_G to the operator output:
//   P_j = d_j (a psi_G);  h_i = J sum_j G_ji P_j;
//   out = c sum_i d_i h_i + V psi_G
// (a = s, c = -1/2 / (J s)), or the weighted transpose for the hermitian form
// (d^T, G_ij, a = w / (J s), c = -1/2 s / w).
//
// One workgroup takes one term and one vector.  A thread keeps up to kGkPoints
// points of the term grid: their D values P_j and the output stay in registers,
// one bracket h_i at a time goes through LDS, and the D derivative columns that
// the three global passes (k_gk_deriv, k_gk_combine, k_gk_out) write and read
// back never exist.  The tables of a term are shared by its vectors, which run
// on one XCD one after the other.
//
// Bound: the G table, D^2 values per point and vector from L2 (six of seven of
// its requests hit), and the 2 D passes over the grid in LDS.  D=6 SG4 L=5, 8
// vectors: 194 us in its three launches, the whole H|psi> 256 us against 425 us
// with the three passes; with the brackets of all modes in LDS at once, and so
// one to four workgroups per CU, this kernel took 215 us.
#include "evr_hterm.hpp"

namespace evr {

template <typename T, int D>
__global__ __launch_bounds__(1024, 4) void k_gk_term(GkArgs<T> a)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int PPT = kGkPoints;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int b = (int)blockIdx.x, slot = b >> 3, v = slot % a.k;
  const int t = a.order[(slot / a.k) * 8 + (b & 7)];
  if (t < 0) return;
  const TermDev &td = a.terms[t];
  const int n = td.nqt;
  const int64_t off = td.off_nq;
  double *sm = reinterpret_cast<double *>(smem_raw);  // the modes' derivative matrices
  int nq[D], st[D], om[D];
  int words = 0;
  {
    int s = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      nq[d] = a.slots[td.slot[d]].nq;
      st[d] = s;
      s *= nq[d];
      om[d] = words;
      words += nq[d] * nq[d];
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    // row q: the nq coefficients of point q
    const double *M = a.D1 + a.slots[td.slot[d]].offD1;
    for (int i = tid; i < nq[d] * nq[d]; i += nt) {
      const int q = i / nq[d], k = i - q * nq[d];
      sm[om[d] + i] = a.trans ? M[k + nq[d] * q] : M[q + nq[d] * k];
    }
  }
  double *sg = sm + words;  // a psi_G, then one bracket after the other
  const T *psi = a.G + v * a.sum_nq + off;
  for (int p = tid; p < n; p += nt) sg[p] = a.ain[off + p] * (double)psi[p];
  __syncthreads();
  int pt[PPT], dig[PPT][D];  // points past the end repeat the first
#pragma unroll
  for (int c = 0; c < PPT; ++c) {
    pt[c] = tid + c * nt < n ? tid + c * nt : 0;
    int rem = pt[c];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int r = fdiv(rem, nq[d], 1.0f / (float)nq[d]);
      dig[c][d] = rem - r * nq[d];
      rem = r;
    }
  }
  // derivatives of the grid in LDS along mode d at the thread's points
  auto deriv = [&](int d, double(&r)[PPT]) {
    const double *m[PPT], *x[PPT];
#pragma unroll
    for (int c = 0; c < PPT; ++c) {
      r[c] = 0.0;
      m[c] = sm + om[d] + dig[c][d] * nq[d];
      x[c] = sg + pt[c] - dig[c][d] * st[d];
    }
#pragma unroll 2
    for (int k = 0; k < nq[d]; ++k)
#pragma unroll
      for (int c = 0; c < PPT; ++c) r[c] = fma(m[c][k], x[c][k * st[d]], r[c]);
  };
  double pj[D][PPT], o[PPT];
#pragma unroll
  for (int d = 0; d < D; ++d) deriv(d, pj[d]);
#pragma unroll
  for (int c = 0; c < PPT; ++c) o[c] = 0.0;
#pragma unroll
  for (int i = 0; i < D; ++i) {
    double h[PPT];
#pragma unroll
    for (int c = 0; c < PPT; ++c) {
      const double *g = a.GG + off + pt[c];
      h[c] = 0.0;
#pragma unroll
      for (int j = 0; j < D; ++j)
        h[c] = fma(g[(int64_t)(a.trans ? j * D + i : i * D + j) * a.sum_nq], pj[j][c], h[c]);
      h[c] *= a.J[off + pt[c]];
    }
    __syncthreads();  // the last reads of sg
#pragma unroll
    for (int c = 0; c < PPT; ++c)
      if (tid + c * nt < n) sg[tid + c * nt] = h[c];
    __syncthreads();
    double r[PPT];
    deriv(i, r);
#pragma unroll
    for (int c = 0; c < PPT; ++c) o[c] += r[c];
  }
#pragma unroll
  for (int c = 0; c < PPT; ++c) {
    const int p = tid + c * nt;
    if (p < n) {
      const int64_t g = off + p;
      const double f = a.wq ? -0.5 * a.s[g] / a.wq[g] : -0.5 / (a.J[g] * a.s[g]);
      a.F[v * a.sum_nq + g] = T(fma(f, o[c], a.V[g] * (double)psi[p]));
    }
  }
}

template <typename T>
hipError_t launch_gk_term(const GkArgs<T> &a, int D, int64_t units, int nt, size_t lds, hipStream_t s)
{
  const int64_t nblk = units * a.k;
  if (nblk <= 0) return hipSuccess;
  // the dispatch grid is counted in work-items in 32 bits
  if (nblk > (int64_t)0xFFFFFFFFu / nt) return hipErrorInvalidConfiguration;
#define EVR_GK(N)                                                                                    \
  case N:                                                                                            \
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gk_term<T, N>),                      \
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                 \
    hipLaunchKernelGGL((k_gk_term<T, N>), dim3((unsigned)nblk), dim3(nt), lds, s, a);                \
    break;
  switch (D) {
    EVR_GK(1) EVR_GK(2) EVR_GK(3) EVR_GK(4) EVR_GK(5) EVR_GK(6) EVR_GK(7) EVR_GK(8) EVR_GK(9)
    default: return hipErrorInvalidValue;
  }
#undef EVR_GK
  return hipGetLastError();
}

template hipError_t launch_gk_term<double>(const GkArgs<double> &, int, int64_t, int, size_t, hipStream_t);
template hipError_t launch_gk_term<float>(const GkArgs<float> &, int, int64_t, int, size_t, hipStream_t);

}  // namespace evr
