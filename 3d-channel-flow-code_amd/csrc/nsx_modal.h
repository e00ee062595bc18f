// nsx_modal.h -- tables of the vertical-mode pressure solve (NSX_REFINE_MODAL):
// built on the host by modal_build_host (nsx_modal.hip), uploaded by the
// context, read by the kernels in nsx_modal_dev.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#define NSX_MODAL_MAXLEV 12
// the 2D hierarchy coarsens to this many nodes or fewer, solved by a dense
// inverse per mode
#define NSX_MODAL_COARSE 96
// damping of the columns' Jacobi sweeps and of the prolongation's smoothing
#define NSX_MODAL_OMEGA 0.8f
#define NSX_MODAL_POMEGA (2.0 / 3.0)
// Columns from which the 2D solves run batched over the modes (one launch per
// sweep over the chip) instead of one block per mode.  The 2D solves of a
// random right-hand side to 1e-13 (two cycles), block per mode against batched, ms:
//   columns     16 layers       48           96           128
//    8,192     2.2 / 4.2    2.3 / 4.7    2.5 / 4.8    2.5 / 4.8
//   16,384     4.4 / 4.9    4.5 / 5.5    4.4 / 5.7    4.7 / 5.7
//   24,576     7.6 / 5.3    7.7 / 6.5    7.7 / 6.5    8.1 / 6.8
//   32,640     9.8 / 5.8    9.7 / 6.9    9.7 / 7.4   10.1 / 7.7
//   65,536    19.8 / 6.8   19.7 / 8.8   20.3 / 10.7  22.4 / 11.4
// A block's time goes with the columns, whatever the number of blocks up to
// 128; the batched form's hardly with the columns (launches).  They cross
// near 18,000 columns at 16 layers and 20,000 to 20,500 at 48 to 128: the line
// lies above them all.
#define NSX_MODAL_BATCH 24576
// blocks of the batched kernels, and the most iterations of a cycle
#define NSX_MB_GRID 1024
#define NSX_MB_MEAN 64
#define NSX_MB_ITERS 60
// a sparse matrix's rows in slices of 64 (one wave): entry e of row r at
// ptr[r / 64] + 64 e + r % 64, every row of a slice padded to the longest
// (index 0, value 0)
struct SellHost {
  int n = 0;
  std::vector<int> ptr, col;
  std::vector<float> val;
};

// a matrix row by row
struct CsrHost {
  int n = 0;
  std::vector<int> ptr, col;
  std::vector<float> val;
};

// host tables
struct ModalHost {
  int N0 = 0, nzi = 0, nc = 0;
  std::vector<double> phi;  // nzi x nzi, phi[k*nzi+m]: component k (interior layer k+1) of mode m
  std::vector<double> mu;   // nzi eigenvalues, ascending
  // the columns' graph: three neighbours and weights (an edge without a
  // neighbour: the column itself, weight 0)
  std::vector<int> nb;     // N0 x 3
  std::vector<double> w;   // N0 x 3
  struct Level {
    int n = 0;
    std::vector<float> diag, area, sabs;  // L's diagonal, the lumped areas, the sum of |off-diagonals|
    SellHost A;   // off-diagonal entries of L (all levels but the columns)
    SellHost R, P;  // restriction to the next level (rows: its nodes), prolongation from it
    CsrHost Ac, Rc, Pc;  // the same three row by row (levels 0 and 1)
  };
  std::vector<Level> levels;  // level 0: the N0 columns
  std::vector<float> cinv;    // nzi dense nc x nc inverses of the coarsest level
};

// tlay[q]: the vertical coupling per unit area between interior layers q and
// q+1 (q = 0..nzi-2); svl[q]: the horizontal couplings' layer factor
// of interior layer q; nbr/ppec: the columns' neighbours (a value >= N0 or < 0
// is a wall) and edge coefficients, N0 x 3.  Returns 0, or -1 with err set.
int modal_build_host(int N0, int nzi, const int *nbr, const double *ppec, const double *area, const double *tlay,
                     const double *svl, ModalHost &H, std::string &err);

// device view (pointers into device memory)
struct SellDev {
  const int *ptr, *col;
  const float *val;
};

struct CsrDev {
  const int *ptr, *col;
  const float *val;
};

// a degree-2 Chebyshev smoother: first = r / (th d), then c1 first + c2 r' / d
struct Cheb {
  float ith, c1, c2;
};

// where a mode's vector lies: LDS (float offset) or the mode's workspace
struct VecLoc {
  int lds;  // 1: in LDS
  int off;  // floats
};

struct ModalLevelDev {
  int n;
  const float *diag, *area;
  SellDev A, R, P;
  CsrDev Ac, Rc, Pc;
  const Cheb *cheb;  // per mode (the levels between the first and the last)
  VecLoc y, t, b;  // solution, gathered work vector, right-hand side
};

// the batched 2D solves' scalars per mode
struct ModeState {
  double rr, r0, rho, target, scale, inv;
  double as;    // alpha x scale
  float beta;
  int act;      // still iterating
};

struct ModalDev {
  int nzi, nlev, nc;
  int N0, N0p;  // columns, and padded to a multiple of 16 (the row length of bh, xh)
  int kt;       // 16-wide tiles of layers (and of modes)
  int mt;       // output tiles a transform block forms (a panel; 0: one, from global memory), and the panels
  int npanel;
  int agrid;    // blocks of the transform kernels along the columns
  int lds2d;    // dynamic LDS of the 2D solve, bytes
  const double *tfwd;  // matrix-core operands of the forward transform, [mode tile][layer tile][lane][4]
  const double *tbwd;  // and of the backward one, [layer tile][mode tile][lane][4]
  const double *mu;    // 16 kt (padding modes: 1)
  const float *cinv;   // the coarsest level's inverses, [m][J][K]
  const int *nb;       // N0 x 3
  const float4 *wa;    // w0, w1, w2, area of every column
  const double *w64, *area64;
  ModalLevelDev lev[NSX_MODAL_MAXLEV];
  VecLoc z0, p[2];     // the columns' further vectors (V in lev[0].y)
  int nwork;           // floats of a mode's workspace
  double *bh, *xh;     // 16 kt x N0p modal right-hand sides (then residuals) and solutions
  double *ap;          // 16 kt x N0p, A p
  float *work;         // nzi x nwork
  double *part;        // npanel x agrid partial sums of the forward transform
  // batched form: bh, xh, ap and the vectors below are node-major, rows of mp
  // modes
  int batched;
  int mp;                    // 16 kt
  float *R, *V, *Z, *W, *P[2];  // the columns' FP32 vectors
  float *y1, *t1, *b1;       // level 1
  float *y2, *b2;            // level 2
  ModeState *ms;             // mp
  double *rpart;             // NSX_MB_MEAN partial sums of mode 0
  double *rpart2;            // NSX_MB_GRID x mp partial sums per mode
  int *nact;                 // per iteration: 1 + the last mode still iterating (0: none)
};
