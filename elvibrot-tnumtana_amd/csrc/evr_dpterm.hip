// H|psi> of one term of two to four modes over the whole device (a
// direct-product basis, or a term beyond one workgroup's LDS) in three passes,
// the same sequence as the mode-by-mode passes of evr_stream.hip
// (BGSG4:2385-2581, OPSG4:1448-1650, BGSG4:2690-2795):
//   first group of modes: psi, its derivatives P_j along the group's modes and
//     K psi (K_i: the part of the operator that acts on mode i alone) on the
//     group's grid, each as a product of 1D matrices (B, D1 B, K B);
//   last group: the tensors on the whole grid, V psi, all P_j, the brackets
//     h_i = sum_j c_ij(q) P_j, and back to the last group's basis at once with
//     W and W D1;
//   first group: W and W D1 on the result and on the group's brackets, summed.
// K_i is c_ii D1_i D1_i of a constant diagonal G (type 10), or F2_ii D2_i +
// F1_i D1_i (type 1); such an operator without cross terms forms no P_j.
//
// Tile: a workgroup holds 2^cbs columns (values of the vector and of the modes
// outside the group) of all points of the group in LDS.  A wave contracts an
// item of 16 outputs for 32 pencils on MFMA (16x16x4): the inputs from LDS, the
// matrix from L1.  In the last group a wave keeps one item of grid points, its
// P_j are used as they are formed and the brackets stay in registers, so
// neither a derivative nor a bracket of the whole grid reaches memory apart
// from those of the first group.
//
// Bound: small terms by the latency of the three launches (3 x 12 functions,
// 2 vectors: H|psi> 23 us, 77 us with 22 mode-by-mode launches; 17 x 23 x 14, 5
// vectors 22 us, before 82 us); large ones by the barriers between the steps of
// the last group, one workgroup of 12 waves per CU (4 x 20 functions, 32
// vectors: 93 + 362 + 104 us, H|psi> 560 us, 827 us before; its MFMA time alone
// is 101 us of the 362).  The same with 8 outputs of 64 pencils per wave on
// scalar coefficients waits for them: 215 + 682 + 123 us.  The matrices in LDS
// instead of L1 change nothing (351 us), tiles of 4 columns cost 170 us more.
#include "evr_dpterm.hpp"

namespace evr {

namespace {

__device__ __forceinline__ int dp_wave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }
__device__ __forceinline__ int dp_lane() { return (int)threadIdx.x & 63; }

// An item's values: element e of a lane is output (lane / 16) + 4 (e % 4) of
// pencil lane % 16 + 16 (e / 4).
struct DpAcc {
  using v4 = double __attribute__((ext_vector_type(4)));
  v4 b[2];
  __device__ __forceinline__ double operator[](int e) const { return b[e >> 2][e & 3]; }
  __device__ __forceinline__ void set(int e, double v) { b[e >> 2][e & 3] = v; }
  __device__ __forceinline__ void clear()
  {
#pragma unroll
    for (int e = 0; e < 8; ++e) set(e, 0.0);
  }
};
// K steps of 4 inputs whose loads are in flight together: as many as the
// registers take beside the values that the last group keeps
constexpr int kDpSteps = 6;
constexpr int kDpStepsLast = 3;

// acc += sum_i M[i ld + o] x[i sx] for the item's outputs (M at its first one)
// and the lane's pencils at x0 and x1
template <int STEPS>
__device__ __forceinline__ void dp_dot(const double *x0, const double *x1, int sx, const double *M, int ld, int nin,
                                       DpAcc &acc)
{
  const int lane = dp_lane(), kr = lane >> 4, ks = (nin + 3) >> 2;
  const double *m = M + (lane & 15);
  for (int s = 0; s < ks; s += STEPS) {
    double am[STEPS], v0[STEPS], v1[STEPS];
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      const int i = 4 * min(s + u, ks - 1) + kr, ix = min(i, nin - 1) * sx;
      am[u] = m[i * ld];  // zero rows past nin
      v0[u] = x0[ix];
      v1[u] = x1[ix];
    }
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
      if (s + u < ks) {
        acc.b[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(am[u], v0[u], acc.b[0], 0, 0, 0);
        acc.b[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(am[u], v1[u], acc.b[1], 0, 0, 0);
      }
  }
}

// the waves' items (tile of 16 outputs, 32 of np pencils): f(first output, the
// lane's pencil of each tile, -1 past np)
template <typename F>
__device__ __forceinline__ void dp_items(int np, int nout, F f)
{
  const int pb = (np + kDpPencils - 1) / kDpPencils, n = pb * ((nout + kDpOut - 1) / kDpOut), nw = (int)blockDim.x >> 6;
  for (int it = dp_wave(); it < n; it += nw) {
    const int ch = it / pb, p = (it - ch * pb) * kDpPencils + (dp_lane() & 15);
    f(ch * kDpOut, p < np ? p : -1, p + 16 < np ? p + 16 : -1);
  }
}

// g(output, pencil, value) for an item's values
template <typename G>
__device__ __forceinline__ void dp_each(const DpAcc &acc, int o0, int nout, int p0, int p1, G g)
{
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int o = o0 + (dp_lane() >> 4) + 4 * (e & 3), p = e < 4 ? p0 : p1;
    if (p >= 0 && o < nout) g(o, p, acc[e]);
  }
}

// Tiles are [point of the group, its first mode fastest][column].
// First mode of two: M (nin -> nout) for each of the nv points of the second.
template <int STEPS>
__device__ __forceinline__ void dp_mode_u(const double *in, double *out, const double *M, int nin, int nout, int nv,
                                          int cbs)
{
  const int cb = 1 << cbs;
  auto at = [&](int p, int n) { return ((n * (p >> cbs)) << cbs) + (p & (cb - 1)); };
  dp_items(nv << cbs, nout, [&](int o0, int p0, int p1) {
    DpAcc acc;
    acc.clear();
    dp_dot<STEPS>(in + at(max(p0, 0), nin), in + at(max(p1, 0), nin), cb, M + o0, dp_pad(nout), nin, acc);
    dp_each(acc, o0, nout, p0, p1, [&](int o, int p, double v) { out[at(p, nout) + (o << cbs)] = v; });
  });
}

// the XCDs (workgroup id modulo 8) take contiguous runs of tiles: neighbours
// share lines of memory
__device__ __forceinline__ int dp_tile(int n)
{
  const int per = (n + 7) >> 3, b = (int)blockIdx.x;
  return (b & 7) * per + (b >> 3);
}

// address of a column in a tensor of L inner values and S points of the group
__device__ __forceinline__ int64_t dp_col(int c, int L, int S)
{
  const int r = c / L;
  return (c - r * L) + (int64_t)L * S * r;
}

// a tile of S points from a tensor of L inner values
__device__ __forceinline__ void dp_load(const DpArgs &a, int c0, int L, int S, const double *src, double *buf)
{
  const int cb = 1 << a.cbs, c = c0 + ((int)threadIdx.x & (cb - 1));
  const double *s = src + dp_col(c < a.ncols ? c : 0, L, S);
  for (int e = threadIdx.x; e < S << a.cbs; e += blockDim.x)
    buf[e] = c < a.ncols ? s[(int64_t)L * (e >> a.cbs)] : 0.0;
}

}  // namespace

// first pass: the first group to its grid
template <int D>
__global__ __launch_bounds__(64 * kDpWaves, 3) void k_dp_first(DpArgs a)
{
  extern __shared__ __align__(16) double sm[];
  constexpr bool TWO = dp_first(D) == 2;
  const int t = dp_tile(a.ntiles);
  if (t >= a.ntiles) return;
  const int cbs = a.cbs, cb = 1 << cbs, c0 = t << cbs, k = a.k;
  const DpMode &mu = a.m[0], &mv = a.m[TWO ? 1 : 0];
  const int nbu = TWO ? mu.nb : 1, nqu = TWO ? mu.nq : 1, ldv = dp_pad(mv.nq);
  const int Sin = nbu * mv.nb, Sout = nqu * mv.nq;
  double *b0 = sm, *b1 = TWO ? sm + (Sin << cbs) : sm;
  {
    const int c = c0 + ((int)threadIdx.x & (cb - 1)), r = c / k, v = c - r * k;
    for (int e = threadIdx.x; e < Sin << cbs; e += blockDim.x) {
      const int pk = c < a.ncols ? a.map[(e >> cbs) + Sin * r] : -1;
      b0[e] = pk >= 0 ? a.X[(int64_t)pk * a.nvec + a.c0 + v] : 0.0;
    }
  }
  __syncthreads();
  // second mode (or the only one) from the tile to dst
  auto land = [&](int M, double *dst, bool add) {
    dp_items(nqu << cbs, mv.nq, [&](int o0, int p0, int p1) {
      DpAcc acc;
      acc.clear();
      dp_dot<kDpSteps>(b1 + max(p0, 0), b1 + max(p1, 0), nqu << cbs, a.tab + M + o0, ldv, mv.nb, acc);
      dp_each(acc, o0, mv.nq, p0, p1, [&](int o, int p, double x) {
        const int c = c0 + (p & (cb - 1));
        if (c >= a.ncols) return;
        double *q = dst + dp_col(c, k, Sout) + (int64_t)k * ((p >> cbs) + nqu * o);
        *q = add ? *q + x : x;
      });
    });
  };
  if (TWO) {
    dp_mode_u<kDpSteps>(b0, b1, a.tab + mu.B, mu.nb, mu.nq, mv.nb, cbs);
    __syncthreads();
  }
  land(mv.B, a.in[0], false);
  if (a.coupled) land(mv.DB, a.in[TWO ? 2 : 1], false);
  if (a.own) land(mv.KB, a.in[3], false);
  if (TWO) {
    if (a.coupled) {
      __syncthreads();
      dp_mode_u<kDpSteps>(b0, b1, a.tab + mu.DB, mu.nb, mu.nq, mv.nb, cbs);
      __syncthreads();
      land(mv.B, a.in[1], false);
    }
    if (a.own) {
      __syncthreads();
      dp_mode_u<kDpSteps>(b0, b1, a.tab + mu.KB, mu.nb, mu.nq, mv.nb, cbs);
      __syncthreads();
      land(mv.B, a.in[3], true);  // the thread's own values of above
    }
  }
}

// second pass: the last group to its grid, the operator, and back
template <int D>
__global__ __launch_bounds__(64 * kDpWaves, 3) void k_dp_last(DpArgs a)
{
  extern __shared__ __align__(16) double sm[];
  constexpr int NA = dp_first(D), U = D - 2, VM = D - 1;  // U: the last group's first mode (D = 4)
  constexpr bool TWO = D - NA == 2;
  const int t = dp_tile(a.ntiles);
  if (t >= a.ntiles) return;
  const int cbs = a.cbs, cb = 1 << cbs, c0 = t << cbs, k = a.k;
  const DpMode &mu = a.m[U], &mv = a.m[VM];
  const int nbu = TWO ? mu.nb : 1, nqu = TWO ? mu.nq : 1;
  const int nbv = mv.nb, nqv = mv.nq, ldq = dp_pad(nqv), ldb = dp_pad(nbv);
  const int L = a.ncols, Sb = nbu * nbv;
  double *b0 = sm, *b1 = sm + ((nqu * nqv) << cbs);
  // the wave's item: 16 grid points of the last mode, two pencils of each lane
  const int np = nqu << cbs, pb = (np + kDpPencils - 1) / kDpPencils, wave = dp_wave();
  const int o0 = wave / pb * kDpOut, q0 = o0 < nqv ? o0 : 0;
  const int pl = wave % pb * kDpPencils + (dp_lane() & 15);
  const int p0 = o0 < nqv && pl < np ? pl : -1, p1 = o0 < nqv && pl + 16 < np ? pl + 16 : -1;
  const int x0 = max(p0, 0), x1 = max(p1, 0);
  // coordinates of the pencils' other modes and of the item's points
  int gp[2];
  double xm[2][VM], xv[4];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int p = b ? x1 : x0;
    int rem = min(c0 + (p & (cb - 1)), L - 1) / k;
    gp[b] = rem;
#pragma unroll
    for (int d = 0; d < NA; ++d) {
      const int r = d == NA - 1 ? 0 : rem / a.m[d].nq, q = rem - r * a.m[d].nq;
      xm[b][d] = a.hasA ? a.x[a.offX[d] + q] : 0.0;
      rem = r;
    }
    if (TWO) xm[b][U] = a.hasA ? a.x[a.offX[U] + (p >> cbs)] : 0.0;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    xv[j] = a.hasA ? a.x[a.offX[VM] + min(q0 + (dp_lane() >> 4) + 4 * j, nqv - 1)] : 0.0;
  int nA = 1;
#pragma unroll
  for (int d = 0; d < NA; ++d) nA *= a.m[d].nq;
  DpAcc h[D], o, P;
  o.clear();
#pragma unroll
  for (int i = 0; i < D; ++i) h[i].clear();
  double *src = b0;  // basis of the last mode, grid of the other
  constexpr int STEPS = TWO ? kDpStepsLast : kDpSteps;
  auto land = [&](int M, DpAcc &acc) {
    dp_dot<STEPS>(src + x0, src + x1, np, a.tab + M + q0, ldq, nbv, acc);
  };
  // brackets from P_j at the wave's points
  auto bracket = [&](int j) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      double g0 = a.C[i * D + j], g1 = g0, gv = 0.0;
      if (a.hasA) {
        const ctab A = a.A + (i * D + j) * D;
#pragma unroll
        for (int m = 0; m < VM; ++m) {
          g0 = fma(A[m], xm[0][m], g0);
          g1 = fma(A[m], xm[1][m], g1);
        }
        gv = A[VM];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) h[i].set(e, fma(fma(gv, xv[e & 3], e < 4 ? g0 : g1), P[e], h[i][e]));
    }
  };
  auto tile_u = [&](int M) {
    if (TWO) {
      __syncthreads();
      dp_mode_u<kDpStepsLast>(b0, b1, a.tab + M, mu.nb, mu.nq, nbv, cbs);
      __syncthreads();
      src = b1;
    }
  };
  dp_load(a, c0, L, Sb, a.in[0], b0);
  if (!TWO) __syncthreads();
  tile_u(mu.B);
  if (a.V) {
    P.clear();
    land(mv.B, P);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int q = min(q0 + (dp_lane() >> 4) + 4 * (e & 3), nqv - 1), qu = (e < 4 ? x0 : x1) >> cbs;
      o.set(e, a.V[gp[e >> 2] + (int64_t)nA * (qu + nqu * q)] * P[e]);
    }
  }
  if (a.own) land(mv.KB, o);
  if (a.coupled) {
    P.clear();
    land(mv.DB, P);
    bracket(VM);
  }
  if (TWO) {
    if (a.coupled) {
      tile_u(mu.DB);
      P.clear();
      land(mv.B, P);
      bracket(U);
    }
    if (a.own) {
      tile_u(mu.KB);
      land(mv.B, o);
    }
  }
  if (a.own) {
    __syncthreads();
    dp_load(a, c0, L, Sb, a.in[3], b0);
    if (!TWO) __syncthreads();
    tile_u(mu.B);
    land(mv.B, o);
  }
  if (a.coupled)
    for (int j = 0; j < NA; ++j) {
      __syncthreads();
      dp_load(a, c0, L, Sb, a.in[1 + j], b0);
      if (!TWO) __syncthreads();
      tile_u(mu.B);
      P.clear();
      land(mv.B, P);
      bracket(j);
    }
  // back: the wave's points to a tile, a chunk of the last mode's functions
  // from it, and with a second mode through a tile again
  auto spread = [&](const DpAcc &v, double *buf) {
    dp_each(v, o0, nqv, p0, p1, [&](int q, int p, double x) { buf[p + np * q] = x; });
  };
  auto spread_b = [&](const DpAcc &v, double *buf) {
    dp_each(v, o0, nbv, p0, p1, [&](int b, int p, double x) { buf[p + np * b] = x; });
  };
  auto from = [&](const double *buf, int M, DpAcc &acc) {
    if (o0 < nbv) dp_dot<STEPS>(buf + x0, buf + x1, np, a.tab + M + o0, ldb, nqv, acc);
  };
  auto store = [&](const DpAcc &v, double *dst) {  // a group of one mode
    dp_each(v, o0, nbv, p0, p1, [&](int b, int p, double x) {
      if (c0 + p < L) dst[c0 + p + (int64_t)L * b] = x;
    });
  };
  // the second mode's functions from one or two tiles (grid of it, basis of the last)
  auto store_u = [&](const double *t0, int M0, const double *t1, int M1, double *dst) {
    auto at = [&](int p) { return ((nqu * (p >> cbs)) << cbs) + (p & (cb - 1)); };
    dp_items(nbv << cbs, nbu, [&](int u0, int e0, int e1) {
      const int y0 = at(max(e0, 0)), y1 = at(max(e1, 0)), ldu = dp_pad(nbu);
      DpAcc acc;
      acc.clear();
      dp_dot<kDpStepsLast>(t0 + y0, t0 + y1, cb, a.tab + M0 + u0, ldu, nqu, acc);
      if (t1) dp_dot<kDpStepsLast>(t1 + y0, t1 + y1, cb, a.tab + M1 + u0, ldu, nqu, acc);
      dp_each(acc, u0, nbu, e0, e1, [&](int u, int p, double x) {
        const int c = c0 + (p & (cb - 1));
        if (c < L) dst[c + (int64_t)L * (u + nbu * (p >> cbs))] = x;
      });
    });
  };
  __syncthreads();
  spread(o, b0);
  if (a.coupled) spread(h[VM], b1);
  __syncthreads();
  P.clear();
  from(b0, mv.W, P);
  if (a.coupled) from(b1, mv.WD, P);
  if (!TWO) {
    store(P, a.out[0]);
  } else {
    __syncthreads();
    spread_b(P, b0);
    if (a.coupled) {
      spread(h[U], b1);
      __syncthreads();
      P.clear();
      from(b1, mv.W, P);
      __syncthreads();
      spread_b(P, b1);
    }
    __syncthreads();
    store_u(b0, mu.W, a.coupled ? b1 : nullptr, mu.WD, a.out[0]);
  }
  if (a.coupled) {
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      __syncthreads();
      spread(h[j], b0);
      __syncthreads();
      P.clear();
      from(b0, mv.W, P);
      if (!TWO) {
        store(P, a.out[1 + j]);
      } else {
        __syncthreads();
        spread_b(P, b0);
        __syncthreads();
        store_u(b0, mu.W, nullptr, 0, a.out[1 + j]);
      }
    }
  }
}

// third pass: the first group back to its basis, into the term rows
template <int D>
__global__ __launch_bounds__(64 * kDpWaves, 3) void k_dp_back(DpArgs a)
{
  extern __shared__ __align__(16) double sm[];
  constexpr bool TWO = dp_first(D) == 2;
  const int t = dp_tile(a.ntiles);
  if (t >= a.ntiles) return;
  const int cbs = a.cbs, cb = 1 << cbs, c0 = t << cbs, k = a.k;
  const DpMode &mu = a.m[0], &mv = a.m[TWO ? 1 : 0];
  const int nbu = TWO ? mu.nb : 1, nqu = TWO ? mu.nq : 1;
  const int nbv = mv.nb, nqv = mv.nq, ldb = dp_pad(nbv), S = nqu * nqv, np = nqu << cbs;
  double *b0 = sm, *b1 = b0 + (S << cbs);
  auto put = [&](int row, int col, double v) {
    const int cc = c0 + col;
    if (cc >= a.ncols) return;
    const int r = cc / k, rp = a.rowpos[row + nbu * nbv * r];
    if (rp >= 0) a.R[(int64_t)rp * a.nvec + a.c0 + (cc - r * k)] = a.w * v;
  };
  // the wave's item of the group's last mode (functions), from the tile in b0
  const int pb = (np + kDpPencils - 1) / kDpPencils, wave = dp_wave();
  const int o0 = wave / pb * kDpOut, pl = wave % pb * kDpPencils + (dp_lane() & 15);
  const int p0 = o0 < nbv && pl < np ? pl : -1, p1 = o0 < nbv && pl + 16 < np ? pl + 16 : -1;
  DpAcc acc;
  auto from = [&](const double *src, int M) {
    dp_load(a, c0, k, S, src, b0);
    __syncthreads();
    if (o0 < nbv) dp_dot<kDpSteps>(b0 + max(p0, 0), b0 + max(p1, 0), np, a.tab + M + o0, ldb, nqv, acc);
    __syncthreads();
  };
  auto spread = [&](double *buf) {
    dp_each(acc, o0, nbv, p0, p1, [&](int o, int p, double x) { buf[p + np * o] = x; });
  };
  acc.clear();
  if (TWO && a.coupled) {
    from(a.out[1], mv.W);
    spread(b1);
    acc.clear();
  }
  from(a.out[0], mv.W);
  if (a.coupled) from(a.out[TWO ? 2 : 1], mv.WD);
  if (!TWO) {
    dp_each(acc, o0, nbv, p0, p1, put);
    return;
  }
  spread(b0);
  __syncthreads();
  auto at = [&](int p) { return ((nqu * (p >> cbs)) << cbs) + (p & (cb - 1)); };
  dp_items(nbv << cbs, nbu, [&](int u0, int p0, int p1) {
    const int x0 = at(max(p0, 0)), x1 = at(max(p1, 0)), ldu = dp_pad(nbu);
    DpAcc acc;
    acc.clear();
    dp_dot<kDpSteps>(b0 + x0, b0 + x1, cb, a.tab + mu.W + u0, ldu, nqu, acc);
    if (a.coupled) dp_dot<kDpSteps>(b1 + x0, b1 + x1, cb, a.tab + mu.WD + u0, ldu, nqu, acc);
    dp_each(acc, u0, nbu, p0, p1, [&](int u, int p, double x) { put(u + nbu * (p >> cbs), p & (cb - 1), x); });
  });
}

hipError_t launch_dp_pass(const DpArgs &a, int D, int pass, int threads, size_t lds, hipStream_t s)
{
  // whole runs of tiles per XCD
  const int64_t nblk = (((int64_t)a.ntiles + 7) >> 3) * 8;
  if (nblk <= 0) return hipSuccess;
  if (nblk > (int64_t)0xFFFFFFFFu / threads) return hipErrorInvalidConfiguration;
#define EVR_DP(K)                                                                                    \
  {                                                                                                  \
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&K), hipFuncAttributeMaxDynamicSharedMemorySize, \
                              (int)lds);                                                             \
    hipLaunchKernelGGL(K, dim3((unsigned)nblk), dim3(threads), lds, s, a);                           \
  }
#define EVR_DPD(N)                                                                                   \
  case N:                                                                                            \
    if (pass == 0) EVR_DP(k_dp_first<N>)                                                             \
    else if (pass == 1) EVR_DP(k_dp_last<N>)                                                         \
    else EVR_DP(k_dp_back<N>)                                                                        \
    break;
  switch (D) {
    EVR_DPD(2) EVR_DPD(3) EVR_DPD(4)
    default: return hipErrorInvalidValue;
  }
#undef EVR_DPD
#undef EVR_DP
  return hipGetLastError();
}

}  // namespace evr
