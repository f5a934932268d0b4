// Records of the three-pass H|psi> of a streamed term (evr_dpterm.hip).
#pragma once
#include "evr_hterm.hpp"

namespace evr {

constexpr int kDpOut = 16;      // outputs of a wave's item: the rows of an MFMA tile
constexpr int kDpPencils = 32;  // pencils of an item: two MFMA tiles
constexpr int kDpWaves = 12;    // waves of a workgroup at most
__host__ __device__ constexpr int dp_pad(int n) { return (n + kDpOut - 1) / kDpOut * kDpOut; }
// modes of the first group (the last group holds one mode, two of four)
constexpr int dp_first(int D) { return D == 2 ? 1 : 2; }

// one mode: its extents and its matrices in the table: per input a row of
// dp_pad(nout) outputs, the inputs padded to 4 (zeros)
struct DpMode {
  int nb, nq;
  int B, DB, KB;  // nb rows -> nq: B, D1 B, K B
  int W, WD;      // nq rows -> nb: W, W D1
};

struct DpArgs {
  int k, nvec, c0;      // vectors of the pass, of the call, the first one
  int cbs;              // log2 of the columns of a tile
  int ncols, ntiles;
  int coupled, own, hasA;
  DpMode m[4];
  const double *tab, *x;  // matrices, grid coordinates
  ctab C, A;            // D x D, D x D x D
  int offX[4];
  const double *V;      // of the term (NULL: none)
  const double *X;      // [nb_packed][nvec]
  const int *map;
  double *in[4];        // psi, P of the first group's modes, own part, on (first grid, last basis)
  double *out[3];       // result, brackets of the first group's modes, the same
  double *R;
  const int *rowpos;
  double w;
};

hipError_t launch_dp_pass(const DpArgs &a, int D, int pass, int threads, size_t lds, hipStream_t s);

}  // namespace evr
