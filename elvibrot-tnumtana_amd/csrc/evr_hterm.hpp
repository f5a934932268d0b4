// Records of the register-block H|psi> kernel (evr_hterm.hip) and its launch.
#pragma once
#include "evr_kernels.hpp"

namespace evr {

// shapes of a group: one or two 1D bases (nb functions on nq points) that a
// thread contracts in registers; any other single mode is kHgGeneric
#define EVR_HG_KINDS(X)                                                                              \
  X(1, 3, 4, 1, 1) X(2, 5, 6, 1, 1) X(3, 7, 8, 1, 1) X(4, 9, 10, 1, 1)                               \
  X(5, 3, 4, 3, 4) X(6, 5, 6, 3, 4) X(7, 3, 4, 5, 6) X(8, 5, 6, 5, 6)                                \
  X(9, 3, 3, 1, 1) X(10, 5, 5, 1, 1) X(11, 7, 7, 1, 1) X(12, 9, 9, 1, 1)                             \
  X(13, 3, 3, 3, 3) X(14, 5, 5, 3, 3) X(15, 3, 3, 5, 5) X(16, 5, 5, 5, 5)
// the rotation of a group (nb x nb matrices) runs as the kind of its square shape
#define EVR_HG_SQUARE(X)                                                                             \
  X(9, 3, 3, 1, 1) X(10, 5, 5, 1, 1) X(11, 7, 7, 1, 1) X(12, 9, 9, 1, 1)                             \
  X(13, 3, 3, 3, 3) X(14, 5, 5, 3, 3) X(15, 3, 3, 5, 5) X(16, 5, 5, 5, 5)
constexpr int kHtModes = 8;   // active modes of a term at most
constexpr int kHgGeneric = 0;
constexpr int kHgSquare = 8;  // kinds 1..8 have the square shape kind + 8

// Words of a coefficient row of na active modes: a value per mode, the
// constant, the value for the pencil mode (even: 16-byte aligned rows).  Per
// active list: the row of h, a row per mode (g_jj), a row per pair i < j (row
// 1 + na + j (j - 1) / 2 + i: g_ij + g_ji), the na x na values a_ijj
// ([j na + i]) and the na values f_i.
__host__ __device__ constexpr int hrow_len(int na) { return (na + 3) & ~1; }
__host__ __device__ constexpr int hcoef_words(int na)
{
  return ((1 + na + na * (na - 1) / 2) * hrow_len(na) + na * na + na + 1) & ~1;
}

struct HGroup {
  int kind;             // shape (EVR_HG_KINDS)
  int nb, nq;           // functions and points of the group
  int n1;               // functions of the faster groups (stride of the group in x)
  int mB[2], mW[2];     // 1D matrices in the pool (row-major): B (nq x nb), W (nb x nq)
  int mI[2], mO[2];     // rotation in (U^T) and out (U), nb x nb
  int pw[2];            // words of the mode's four matrices (B first, contiguous)
  int mP[2], mQ[2];     // B and W without the rotation (the transforms)
};

// One term.  Active positions (modes whose P, Q, R do not vanish) in the
// order of the coefficient rows; for pencils of more than one function the
// pencil mode comes first.
struct HTerm {  // sizeof: a multiple of 8
  int64_t off_nb, off_vq;  // term rows (map, rowpos), first value of V
  double w;
  int nbt, na, ng, g0;     // functions, active modes, groups and the first of them
  int nbp;                 // functions per pencil: 1 or 3
  int nm;                  // M arrays held in LDS at a time
  int fw, lC;              // LDS words of the factors and coefficient rows, first of the rows
  int wA, wB;              // words per vector of the two V buffers
  int nbO, QO, nO, nOm;    // slabbed V part: functions and points of the outer groups, groups, modes
  int nbI;                 // functions of the inner modes (nbt / nbO)
  int ngen;                // groups of kind kHgGeneric
  int oB[4], oW[4], onb[4], onq[4];  // matrices and extents of the outer modes
  int coef;                // first coefficient row in the table (hrow_len)
  int nb[kMaxDev], st[kMaxDev];      // functions and stride of the active modes
  int gF[kMaxDev], lF[kMaxDev];      // their factors: in the pool, in LDS
  float rst[kMaxDev], rnb[kMaxDev];  // 1 / st, 1 / nb
};

// Tables read at wave-uniform addresses live in the constant address space:
// their loads are scalar whatever the kernel stores in between.
#ifndef EVR_CONST
#define EVR_CONST __attribute__((address_space(4)))
#endif
using ctab = const double EVR_CONST *;

// One term of the basis <-> grid transforms.  The full grid point p = pl + Pl
// ph splits into the first nlow modes (pl) and the others (ph); each side into
// the points r of its modes with more than one function and the points c of
// its one-function modes, pl = Rl-part + Cl-part.
struct XTerm {  // sizeof: a multiple of 8
  int64_t off_nb, off_nq;  // term rows, first point of the term grid
  double w;                // weight of the G->B scatter (0 below 1e-6, BGSG4:1004)
  int nbt, nqt, nvq;       // functions, points, points of the modes with more than one function
  int ng, g0;              // groups and the first of them
  int nlow, D;             // modes of the low part, modes
  int Pl, Ph, Rl, Rh;      // points of the low and high parts, of their r parts
  int wA, wB;              // LDS words of the two tensor buffers, B->G
  int uA, uB;              // the same, G->B
  int nq[kMaxDev];
  int one[kMaxDev];        // one-function modes: offset of B (nq x 1) in the pool, W (1 x nq) follows; -1 else
};

struct XArgs {
  int nvec;
  const int EVR_CONST *order;      // terms of the workgroups
  const XTerm EVR_CONST *terms;
  const HGroup EVR_CONST *groups;
  ctab pool;
  const double *pool1;     // B and W of the one-function modes
  const int *map, *rowpos;
  const double *X;         // B->G: packed block [function][vector]
  double *G;               // B->G: grid columns
  const double *Gin;       // G->B: grid columns
  double *R;               // G->B: term rows [row][vector]
  int64_t gld;             // column stride of the grid
};

// One launch.  The pointers are read from the argument block where they are
// used, so they do not hold scalar registers over the whole kernel.
struct HArgs {
  int lv;                  // NV = 1 << lv
  int nvec;
  int hasV, hasKeo, hasA, hasM;
  const int EVR_CONST *order;      // terms of the workgroups (-1 = padding)
  const HTerm EVR_CONST *terms;
  const HGroup EVR_CONST *groups;
  ctab pool;               // 1D matrices
  const double *fpool;     // factor rows
  const double *coef;      // coefficient rows
  const int *map, *rowpos;
  const double *V, *X;
  double *R;
};

// Grid form of type 10 with G, J, s per point, one term per workgroup
// (evr_gkterm.hip); psi_G, out in T, tables FP64.
template <typename T>
struct GkArgs {
  int k;                   // vectors
  int trans;               // the weighted transpose
  const int *order;        // terms of the workgroups (-1 = padding)
  const TermDev *terms;
  const SlotDev *slots;
  const double *D1, *ain, *J, *GG, *s, *V, *wq;
  const T *G;
  T *F;
  int64_t sum_nq;
};
// points a thread holds, their D derivatives in registers: with 4 the D=6 kernel
// spills 164 registers of its 128 (726 us for the H|psi> of D=6 L=5 with 8
// vectors, 285 us with 2)
constexpr int kGkPoints = 2;
// modes the kernel is built for: with ten and more it spills 76 to 179
// registers and terms of few points run slower than the three passes (8 vectors:
// D=10 L=5 law 1,1,1,1 721 against 659 us, D=12 L=4 708 against 558 us; D=8 L=5
// 242 against 307 us)
constexpr int kGkModes = 9;
template <typename T>
hipError_t launch_gk_term(const GkArgs<T> &a, int D, int64_t units, int nt, size_t lds, hipStream_t s);

// most threads and LDS words of a transform workgroup; high r points a wave of
// the G->B contraction takes at a time
constexpr int kXThreads = 256;
constexpr int kXRows = 2;
size_t xform_words(const XTerm &t, bool b2g);
// basis -> grid or grid -> basis on n terms x nvec vectors in workgroups of nt threads (whole waves)
hipError_t launch_xform(const XArgs &a, bool b2g, int64_t nterms, int nt, size_t lds, hipStream_t s);

// k_hterm on nblk workgroups of nt threads
hipError_t launch_hterm(const HArgs &a, int64_t nblk, int nt, size_t lds, hipStream_t s);

}  // namespace evr
