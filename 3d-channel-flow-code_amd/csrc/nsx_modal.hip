// nsx_modal.hip -- host set-up of the vertical-mode pressure solve
// (NSX_REFINE_MODAL).
//
// The PPE operator of the prismatic sigma grid is a Kronecker sum: a
// horizontal coupling between columns i and j at layer k is ppec(i,j)
// dsigv(k-1), a vertical one between layers k and k+1 of column i is area(i)
// t(k) (t = 1/dsig, none at the top and bottom, which every product mirrors),
// and the diagonal closes every row to zero (PDE_center, PDE.F90:8-135).  So
// -A = L (x) S + D (x) T with L the weighted graph Laplacian of the columns, D
// = diag(area), S = diag(dsigv) and T the layers' 1D Laplacian.  The
// generalized eigenvectors Phi of (T, S) (Phi^T S Phi = I, Phi^T T Phi =
// diag(mu)) split -A y = r into one 2D problem per vertical mode m, (L + mu_m
// D) yh_m = (Phi^T r)_m with y = Phi yh.  The solve transforms a residual
// once, solves every mode's 2D problem by conjugate gradients of its own, and
// transforms back; the 2D preconditioner is a V-cycle of smoothed-aggregation
// multigrid on the column graph.  This file builds the tables on the host: the
// modes, the hierarchy, the coarsest level's inverses.  The kernels are in
// nsx_modal_dev.hip.
//
// The hierarchy is built from L alone and serves every mode: aggregates are a
// node and its neighbours (roots with no aggregated neighbour first, the rest
// join their strongest neighbour's), the prolongation is the piecewise
// constant one smoothed by a damped Jacobi step (P = (I - omega D_L^-1 L) P0,
// rows summing to one), the coarse Laplacian is P^T L P and the coarse areas
// are P^T area (the mass matrix P^T D P lumped to its row sums).  On a
// 65,536-column channel the levels hold 65,536, 13,763, 1,051 and 46 nodes
// and conjugate gradients take 15 iterations for 1e-6 on mode 0 and 6 to 14
// on the others; piecewise-constant prolongation takes 58 and 9 to 44.
#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "nsx_modal.h"

namespace {

// eigenvalues d and orthonormal eigenvectors of the symmetric tridiagonal
// n x n matrix with diagonal d and off-diagonal e (e[i] couples i and i+1),
// by QR iterations with Wilkinson's shift and deflation at negligible
// couplings; v[m*n+k] is component k of vector m.  Returns false if an
// eigenvalue does not settle.
bool tridiag_eigen(int n, std::vector<double> &d, std::vector<double> e, std::vector<double> &v) {
  v.assign((size_t)n * n, 0.0);
  for (int i = 0; i < n; ++i) v[(size_t)i * n + i] = 1.0;
  e.resize(n, 0.0);
  int hi = n - 1;
  for (int sweep = 0; hi > 0; ++sweep) {
    if (sweep > 60 * n) return false;
    auto small = [&](int i) { return std::fabs(e[i]) <= 1e-17 * (std::fabs(d[i]) + std::fabs(d[i + 1])); };
    if (small(hi - 1)) {
      e[hi - 1] = 0.0;
      --hi;
      continue;
    }
    int lo = hi - 1;
    while (lo > 0 && !small(lo - 1)) --lo;
    if (lo > 0) e[lo - 1] = 0.0;
    // the eigenvalue of the trailing 2 x 2 block nearer to d[hi]
    const double half = 0.5 * (d[hi - 1] - d[hi]), c2 = e[hi - 1] * e[hi - 1];
    const double root = std::hypot(half, e[hi - 1]);
    const double shift = d[hi] - c2 / (half + (half >= 0 ? root : -root));
    // chase the bulge of the shifted step's first rotation down the block
    double x = d[lo] - shift, y = e[lo];
    for (int i = lo; i < hi; ++i) {
      const double h = std::hypot(x, y);
      const double c = h > 0 ? x / h : 1.0, s = h > 0 ? y / h : 0.0;
      if (i > lo) e[i - 1] = h;
      const double a = d[i], b = d[i + 1], f = e[i];
      d[i] = c * c * a + 2 * c * s * f + s * s * b;
      d[i + 1] = s * s * a - 2 * c * s * f + c * c * b;
      e[i] = c * s * (b - a) + (c * c - s * s) * f;
      if (i + 1 < hi) {
        x = e[i];
        y = s * e[i + 1];
        e[i + 1] *= c;
      }
      double *p = &v[(size_t)i * n], *q = p + n;
      for (int k = 0; k < n; ++k) {
        const double pk = p[k], qk = q[k];
        p[k] = c * pk + s * qk;
        q[k] = c * qk - s * pk;
      }
    }
  }
  return true;
}

// inverse of the n x n matrix a (row-major) by Gauss-Jordan elimination with
// partial pivoting; false when it is singular to working precision
bool invert(int n, std::vector<double> a, std::vector<double> &inv) {
  inv.assign((size_t)n * n, 0.0);
  for (int i = 0; i < n; ++i) inv[(size_t)i * n + i] = 1.0;
  for (int c = 0; c < n; ++c) {
    int piv = c;
    for (int r = c + 1; r < n; ++r)
      if (std::fabs(a[(size_t)r * n + c]) > std::fabs(a[(size_t)piv * n + c])) piv = r;
    if (!(std::fabs(a[(size_t)piv * n + c]) > 0.0)) return false;
    if (piv != c)
      for (int k = 0; k < n; ++k) {
        std::swap(a[(size_t)c * n + k], a[(size_t)piv * n + k]);
        std::swap(inv[(size_t)c * n + k], inv[(size_t)piv * n + k]);
      }
    const double d = 1.0 / a[(size_t)c * n + c];
    for (int k = 0; k < n; ++k) {
      a[(size_t)c * n + k] *= d;
      inv[(size_t)c * n + k] *= d;
    }
    for (int r = 0; r < n; ++r) {
      if (r == c) continue;
      const double f = a[(size_t)r * n + c];
      if (f == 0.0) continue;
      for (int k = 0; k < n; ++k) {
        a[(size_t)r * n + k] -= f * a[(size_t)c * n + k];
        inv[(size_t)r * n + k] -= f * inv[(size_t)c * n + k];
      }
    }
  }
  return true;
}

// the off-diagonal entries of a symmetric matrix in CSR, its diagonal and the
// nodes' areas
struct Graph {
  int n = 0;
  std::vector<int> ptr, col;
  std::vector<double> a, diag, area;
};

// a rectangular matrix in CSR
struct Csr {
  int n = 0, m = 0;
  std::vector<int> ptr, col;
  std::vector<double> val;
};

// one row gathered from (column, value) pairs in any order: `slot` holds the
// place of each column in the row, -1 when absent (left so again by clear)
struct RowSum {
  std::vector<int> slot, col;
  std::vector<double> val;
  explicit RowSum(int m) : slot(m, -1) {}
  void add(int c, double v) {
    if (slot[c] < 0) {
      slot[c] = (int)col.size();
      col.push_back(c);
      val.push_back(v);
    } else {
      val[slot[c]] += v;
    }
  }
  void clear() {
    for (int c : col) slot[c] = -1;
    col.clear();
    val.clear();
  }
};

Csr transpose(const Csr &A) {
  Csr T;
  T.n = A.m;
  T.m = A.n;
  T.ptr.assign(A.m + 1, 0);
  for (int c : A.col) ++T.ptr[c + 1];
  for (int i = 0; i < A.m; ++i) T.ptr[i + 1] += T.ptr[i];
  T.col.resize(A.col.size());
  T.val.resize(A.col.size());
  std::vector<int> at(T.ptr.begin(), T.ptr.end() - 1);
  for (int i = 0; i < A.n; ++i)
    for (int q = A.ptr[i]; q < A.ptr[i + 1]; ++q) {
      T.col[at[A.col[q]]] = i;
      T.val[at[A.col[q]]++] = A.val[q];
    }
  return T;
}

// aggregates: a node none of whose neighbours is taken seeds one with all of
// them; every other node joins the aggregate of the taken neighbour it is
// coupled to most strongly
std::vector<int> aggregate(const Graph &G, int &na) {
  std::vector<int> agg(G.n, -1);
  na = 0;
  for (int i = 0; i < G.n; ++i) {
    bool free = agg[i] < 0;
    for (int q = G.ptr[i]; free && q < G.ptr[i + 1]; ++q) free = agg[G.col[q]] < 0;
    if (!free) continue;
    agg[i] = na;
    for (int q = G.ptr[i]; q < G.ptr[i + 1]; ++q) agg[G.col[q]] = na;
    ++na;
  }
  std::vector<int> out = agg;
  for (int i = 0; i < G.n; ++i) {
    if (agg[i] >= 0) continue;
    double best = 0.0;
    int at = -1;
    for (int q = G.ptr[i]; q < G.ptr[i + 1]; ++q)
      if (agg[G.col[q]] >= 0 && (at < 0 || -G.a[q] > best)) {
        best = -G.a[q];
        at = agg[G.col[q]];
      }
    out[i] = at >= 0 ? at : na++;
  }
  return out;
}

// (I - omega D^-1 L) P0
Csr smoothed_prolongation(const Graph &G, const std::vector<int> &agg, int na) {
  Csr P;
  P.n = G.n;
  P.m = na;
  P.ptr.assign(1, 0);
  RowSum row(na);
  for (int i = 0; i < G.n; ++i) {
    const double f = G.diag[i] > 0.0 ? NSX_MODAL_POMEGA / G.diag[i] : 0.0;
    row.add(agg[i], 1.0 - f * G.diag[i]);
    for (int q = G.ptr[i]; q < G.ptr[i + 1]; ++q) row.add(agg[G.col[q]], -f * G.a[q]);
    P.col.insert(P.col.end(), row.col.begin(), row.col.end());
    P.val.insert(P.val.end(), row.val.begin(), row.val.end());
    P.ptr.push_back((int)P.col.size());
    row.clear();
  }
  return P;
}

// P^T L P with the diagonal that closes its rows to zero, and P^T area
Graph galerkin(const Graph &G, const Csr &P, const Csr &R) {
  Graph C;
  C.n = P.m;
  C.area.assign(C.n, 0.0);
  C.diag.assign(C.n, 0.0);
  C.ptr.assign(1, 0);
  // L P, row by row
  Csr LP;
  LP.n = G.n;
  LP.m = P.m;
  LP.ptr.assign(1, 0);
  RowSum row(P.m);
  for (int i = 0; i < G.n; ++i) {
    for (int q = P.ptr[i]; q < P.ptr[i + 1]; ++q) row.add(P.col[q], G.diag[i] * P.val[q]);
    for (int e = G.ptr[i]; e < G.ptr[i + 1]; ++e)
      for (int q = P.ptr[G.col[e]]; q < P.ptr[G.col[e] + 1]; ++q) row.add(P.col[q], G.a[e] * P.val[q]);
    LP.col.insert(LP.col.end(), row.col.begin(), row.col.end());
    LP.val.insert(LP.val.end(), row.val.begin(), row.val.end());
    LP.ptr.push_back((int)LP.col.size());
    row.clear();
  }
  for (int J = 0; J < C.n; ++J) {
    for (int q = R.ptr[J]; q < R.ptr[J + 1]; ++q) {
      const int i = R.col[q];
      C.area[J] += R.val[q] * G.area[i];
      for (int e = LP.ptr[i]; e < LP.ptr[i + 1]; ++e) row.add(LP.col[e], R.val[q] * LP.val[e]);
    }
    for (size_t q = 0; q < row.col.size(); ++q)
      if (row.col[q] != J) {
        C.col.push_back(row.col[q]);
        C.a.push_back(row.val[q]);
        C.diag[J] -= row.val[q];
      }
    C.ptr.push_back((int)C.col.size());
    C.area[J] = std::max(C.area[J], 0.0);
    row.clear();
  }
  return C;
}

SellHost to_sell(int n, const std::vector<int> &ptr, const std::vector<int> &col, const std::vector<double> &val) {
  SellHost S;
  S.n = n;
  S.ptr.assign(1, 0);
  for (int s = 0; s < n; s += 64) {
    int len = 0;
    for (int r = s; r < std::min(n, s + 64); ++r) len = std::max(len, ptr[r + 1] - ptr[r]);
    S.ptr.push_back(S.ptr.back() + 64 * len);
  }
  S.col.assign(S.ptr.back(), 0);
  S.val.assign(S.ptr.back(), 0.0f);
  for (int r = 0; r < n; ++r)
    for (int q = ptr[r]; q < ptr[r + 1]; ++q) {
      const size_t at = (size_t)S.ptr[r / 64] + 64 * (size_t)(q - ptr[r]) + r % 64;
      S.col[at] = col[q];
      S.val[at] = (float)val[q];
    }
  return S;
}

CsrHost to_csr(int n, const std::vector<int> &ptr, const std::vector<int> &col, const std::vector<double> &val) {
  return {n, ptr, col, std::vector<float>(val.begin(), val.end())};
}

}  // namespace

int modal_build_host(int N0, int nzi, const int *nbr, const double *ppec, const double *area, const double *tlay,
                     const double *svl, ModalHost &H, std::string &err) {
  if (nzi < 1 || N0 < 2) {
    err = "vertical-mode solve: empty mesh";
    return -1;
  }
  H.N0 = N0;
  H.nzi = nzi;
  // vertical modes: C = S^-1/2 T S^-1/2, Phi = S^-1/2 Y
  std::vector<double> rs(nzi), d(nzi, 0.0), e(nzi, 0.0), Y;
  for (int q = 0; q < nzi; ++q) {
    if (!(svl[q] > 0.0)) {
      err = "vertical-mode solve: a layer with dsigv <= 0";
      return -1;
    }
    rs[q] = 1.0 / std::sqrt(svl[q]);
  }
  for (int q = 0; q + 1 < nzi; ++q) {
    d[q] += tlay[q] * rs[q] * rs[q];
    d[q + 1] += tlay[q] * rs[q + 1] * rs[q + 1];
    e[q] = -tlay[q] * rs[q] * rs[q + 1];
  }
  if (!tridiag_eigen(nzi, d, e, Y)) {
    err = "vertical-mode solve: the vertical eigenproblem did not converge";
    return -1;
  }
  std::vector<int> order(nzi);
  for (int m = 0; m < nzi; ++m) order[m] = m;
  std::sort(order.begin(), order.end(), [&](int a, int b) { return d[a] < d[b]; });
  H.mu.resize(nzi);
  H.phi.assign((size_t)nzi * nzi, 0.0);
  for (int m = 0; m < nzi; ++m) {
    H.mu[m] = std::max(d[order[m]], 0.0);
    for (int k = 0; k < nzi; ++k) H.phi[(size_t)k * nzi + m] = rs[k] * Y[(size_t)order[m] * nzi + k];
  }
  // T has the constants as its null vector (Neumann at both ends): mode 0 is
  // exactly constant
  {
    double s = 0.0;
    for (int k = 0; k < nzi; ++k) s += svl[k];
    H.mu[0] = 0.0;
    for (int k = 0; k < nzi; ++k) H.phi[(size_t)k * nzi] = 1.0 / std::sqrt(s);
  }
  // level 0: the columns, edges to interior neighbours, weights made
  // symmetric (the average of the two directions)
  H.nb.resize((size_t)N0 * 3);
  H.w.assign((size_t)N0 * 3, 0.0);
  Graph G;
  G.n = N0;
  G.area.assign(area, area + N0);
  G.diag.assign(N0, 0.0);
  G.ptr.assign(1, 0);
  RowSum row(N0);
  for (int i = 0; i < N0; ++i) {
    for (int j = 0; j < 3; ++j) {
      const int n = nbr[i * 3 + j];
      H.nb[(size_t)i * 3 + j] = i;
      if (n < 0 || n >= N0 || n == i) continue;
      // the neighbour's weights back towards i, shared by i's edges to it (the
      // sums over a pair's edges agree both ways, whatever their numbers)
      double back = 0.0;
      int to = 0;
      for (int q = 0; q < 3; ++q) {
        if (nbr[n * 3 + q] == i) back += ppec[n * 3 + q];
        if (nbr[i * 3 + q] == n) ++to;
      }
      const double w = 0.5 * (ppec[i * 3 + j] + back / to);
      H.nb[(size_t)i * 3 + j] = n;
      H.w[(size_t)i * 3 + j] = w;
      G.diag[i] += w;
      row.add(n, -w);
    }
    G.col.insert(G.col.end(), row.col.begin(), row.col.end());
    G.a.insert(G.a.end(), row.val.begin(), row.val.end());
    G.ptr.push_back((int)G.col.size());
    row.clear();
  }
  H.levels.clear();
  for (;;) {
    H.levels.emplace_back();
    ModalHost::Level &o = H.levels.back();
    o.n = G.n;
    o.diag.assign(G.diag.begin(), G.diag.end());
    o.area.assign(G.area.begin(), G.area.end());
    o.sabs.assign(G.n, 0.0f);
    for (int i = 0; i < G.n; ++i) {
      double s = 0.0;
      for (int q = G.ptr[i]; q < G.ptr[i + 1]; ++q) s += std::fabs(G.a[q]);
      o.sabs[i] = (float)s;
    }
    if (H.levels.size() > 1) o.A = to_sell(G.n, G.ptr, G.col, G.a);
    if (H.levels.size() == 2) o.Ac = to_csr(G.n, G.ptr, G.col, G.a);
    if (G.n <= NSX_MODAL_COARSE || (int)H.levels.size() == NSX_MODAL_MAXLEV) break;
    int na = 0;
    const std::vector<int> agg = aggregate(G, na);
    if (na > 0.9 * G.n) break;
    const Csr P = smoothed_prolongation(G, agg, na), R = transpose(P);
    o.P = to_sell(P.n, P.ptr, P.col, P.val);
    o.R = to_sell(R.n, R.ptr, R.col, R.val);
    if (H.levels.size() <= 2) {
      o.Pc = to_csr(P.n, P.ptr, P.col, P.val);
      o.Rc = to_csr(R.n, R.ptr, R.col, R.val);
    }
    G = galerkin(G, P, R);
  }
  // the coarsest level's inverses, one per mode; the Neumann mode (mu = 0, L
  // singular with the constant null vector) by the inverse with node 0
  // pinned, between projections onto zero mean
  const int nc = G.n;
  if (nc > 1024) {
    err = "vertical-mode solve: the column graph does not coarsen";
    return -1;
  }
  H.nc = nc;
  H.cinv.assign((size_t)nzi * nc * nc, 0.0f);
  std::vector<double> A((size_t)nc * nc), inv;
  for (int m = 0; m < nzi; ++m) {
    std::fill(A.begin(), A.end(), 0.0);
    for (int i = 0; i < nc; ++i) {
      for (int q = G.ptr[i]; q < G.ptr[i + 1]; ++q) A[(size_t)i * nc + G.col[q]] += G.a[q];
      A[(size_t)i * nc + i] += G.diag[i] + H.mu[m] * G.area[i];
    }
    if (m > 0) {
      if (!invert(nc, A, inv)) {
        err = "vertical-mode solve: singular coarse operator";
        return -1;
      }
    } else if (nc > 1) {
      std::vector<double> B((size_t)(nc - 1) * (nc - 1));
      for (int i = 1; i < nc; ++i)
        for (int j = 1; j < nc; ++j) B[(size_t)(i - 1) * (nc - 1) + (j - 1)] = A[(size_t)i * nc + j];
      std::vector<double> Bi;
      if (!invert(nc - 1, B, Bi)) {
        err = "vertical-mode solve: singular coarse operator";
        return -1;
      }
      std::vector<double> Gm((size_t)nc * nc, 0.0);
      for (int i = 1; i < nc; ++i)
        for (int j = 1; j < nc; ++j) Gm[(size_t)i * nc + j] = Bi[(size_t)(i - 1) * (nc - 1) + (j - 1)];
      // inv = P Gm P, P = I - 1 1^T / nc
      std::vector<double> rowm(nc, 0.0), colm(nc, 0.0);
      double all = 0.0;
      for (int i = 0; i < nc; ++i)
        for (int j = 0; j < nc; ++j) {
          rowm[i] += Gm[(size_t)i * nc + j] / nc;
          colm[j] += Gm[(size_t)i * nc + j] / nc;
          all += Gm[(size_t)i * nc + j] / ((double)nc * nc);
        }
      inv.assign((size_t)nc * nc, 0.0);
      for (int i = 0; i < nc; ++i)
        for (int j = 0; j < nc; ++j) inv[(size_t)i * nc + j] = Gm[(size_t)i * nc + j] - rowm[i] - colm[j] + all;
    } else {
      inv.assign(1, 0.0);
    }
    for (size_t q = 0; q < (size_t)nc * nc; ++q) H.cinv[(size_t)m * nc * nc + q] = (float)inv[q];
  }
  return 0;
}
