// nsx_modal_dev.hip -- kernels of the vertical-mode pressure solve
// (NSX_REFINE_MODAL; the method and its tables: nsx_modal.hip).
//
// One cycle of the solve, from the FP64 residual r = b - A x:
//   k_modal_fwd   bh_m = (Phi^T r)_m, an FP64 GEMM of the columns against the
//                 mode table on the matrix cores (v_mfma_f64_16x16x4_f64)
//   k_modal_2d    (L + mu_m D) xh_m = bh_m, one block per mode
//   k_modal_bwd   x -= Phi xh, the same GEMM transposed
//   k_modal_true, k_modal_check (nsx_bicgstab.hip)  the next residual, the reference's
//                 stopping rule
// Everything that x sees is FP64; FP32 is the 2D preconditioner's.  The modes
// are independent, so no block waits for another inside a cycle.
#include "nsx_kernels.h"

typedef double f64x4 __attribute__((ext_vector_type(4)));

// --- the transforms.  A wave forms a 16 x 16 tile of the result per output
// tile: D[i][j] += A[i][k] B[k][j] with A[i][k] from lane i + 16 k, B[k][j]
// from lane j + 16 k, and D[i][j] in lane j + 16 (i mod 4), register i / 4.
// The sum over k may run in any order, so step q of layer (mode) tile t takes
// k = 16 t + 4 (lane / 16) + q: a lane reads four consecutive layers.  The
// table's operands are laid out by the host so that a lane's four are one
// 32-byte run in LDS; a block holds the table's panel of MT output tiles (at
// 96 layers all six, 72 KB: two blocks a CU; npanel > 1 where the whole table
// passes the LDS).  MT = 0: one output tile a block whose operands come from
// global memory, for tables of which not one tile fits (more than 1,264
// layers); the LDS form stays the one wherever it fits.
constexpr int MODAL_TB = 256;

template <int MT>
__device__ inline const double *lds_panel(const double *src, int kt) {
  if constexpr (MT == 0) return src;
  extern __shared__ __align__(16) unsigned char nsx_dyn_lds[];
  double2 *dst = reinterpret_cast<double2 *>(nsx_dyn_lds);
  const double2 *s = reinterpret_cast<const double2 *>(src);
  const int n = MT * kt * 128;
#pragma unroll 4
  for (int q = threadIdx.x; q < n; q += MODAL_TB) dst[q] = s[q];
  __syncthreads();
  return reinterpret_cast<const double *>(nsx_dyn_lds);
}

// four consecutive interior layers k .. k+3 of the column at p (its first
// interior layer), zero past the last; the interior starts one slot into a
// column, so the runs are 8-byte aligned
__device__ inline void load_layers(const double *p, int k, int nzi, bool ok, double (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = (ok && k + q < nzi) ? p[k + q] : 0.0;
}

// NODE: bh is node-major (the batched 2D solves): the operands change places,
// and so do D's rows and columns
template <int MT, bool NODE>
__global__ __launch_bounds__(MODAL_TB) void k_modal_fwd(Geo g, ModalDev M, const double *r, const SolverState *st) {
  if (st->done) return;
  constexpr int NT = MT ? MT : 1;
  const int kt = M.kt, nzi = M.nzi, m0 = 16 * NT * (int)blockIdx.y;
  const double *tab = lds_panel<MT>(M.tfwd + (size_t)blockIdx.y * NT * kt * 256, kt);
  const int lane = threadIdx.x & 63, j = lane & 15, gq = lane >> 4;
  const int ntile = M.N0p >> 4, stride = gridDim.x * (MODAL_TB / 64);
  double sum[1] = {0.0};
  for (int tile = blockIdx.x * (MODAL_TB / 64) + (threadIdx.x >> 6); tile < ntile; tile += stride) {
    const int c = 16 * tile + j;
    const bool ok = c < g.N0;
    const double *src = r + (size_t)(ok ? c : 0) * g.NS + 1;
    f64x4 acc[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
    double b[4], bn[4];
    load_layers(src, 4 * gq, nzi, ok, b);
    for (int t = 0; t < kt; ++t) {
      if (t + 1 < kt) load_layers(src, 16 * (t + 1) + 4 * gq, nzi, ok, bn);
      const double *a = tab + ((size_t)t * 64 + lane) * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < NT; ++m)
          acc[m] = NODE ? __builtin_amdgcn_mfma_f64_16x16x4f64(b[q], a[(size_t)m * kt * 256 + q], acc[m], 0, 0, 0)
                        : __builtin_amdgcn_mfma_f64_16x16x4f64(a[(size_t)m * kt * 256 + q], b[q], acc[m], 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) b[q] = bn[q];
    }
    if (NODE) {
      // lanes j: 16 consecutive modes of one column (the padding modes' are 0)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        double *dst = M.bh + (size_t)(16 * tile + gq + 4 * q) * M.mp + m0 + j;
#pragma unroll
        for (int m = 0; m < NT; ++m) {
          if (m0 + 16 * m < M.mp) dst[16 * m] = acc[m][q];
          sum[0] += acc[m][q] * acc[m][q];
        }
      }
      continue;
    }
    // lanes j: 16 consecutive columns of one mode, a 128-byte run
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int mode = m0 + 16 * m + gq + 4 * q;
        if (mode >= nzi) continue;
        M.bh[(size_t)mode * M.N0p + c] = acc[m][q];
        sum[0] += acc[m][q] * acc[m][q];
      }
  }
  write_partials<1, MODAL_TB>(sum, M.part + (size_t)blockIdx.y * gridDim.x);
}

template <int MT, bool NODE>
__global__ __launch_bounds__(MODAL_TB) void k_modal_bwd(Geo g, ModalDev M, double *x, SolverState *st) {
  if (st->done) return;
  constexpr int NT = MT ? MT : 1;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    if (st->mp_pass == 0) st->m_first = st->m_cyc;
    st->m_iters += st->m_cyc;
    st->m_cyc = 0;
    st->mp_pass += 1;
  }
  const int kt = M.kt, nzi = M.nzi, l0 = 16 * NT * (int)blockIdx.y;
  const double *tab = lds_panel<MT>(M.tbwd + (size_t)blockIdx.y * NT * kt * 256, kt);
  const int lane = threadIdx.x & 63, j = lane & 15, gq = lane >> 4;
  const int ntile = M.N0p >> 4, stride = gridDim.x * (MODAL_TB / 64);
  for (int tile = blockIdx.x * (MODAL_TB / 64) + (threadIdx.x >> 6); tile < ntile; tile += stride) {
    f64x4 acc[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
    // xh's padding modes and columns are zero
    const double *src = NODE ? M.xh + (size_t)(16 * tile + j) * M.mp + 4 * gq
                             : M.xh + (size_t)(4 * gq) * M.N0p + 16 * tile + j;
    const size_t step = NODE ? 1 : M.N0p;
    double a[4], an[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = src[q * step];
    for (int t = 0; t < kt; ++t) {
      if (t + 1 < kt)
#pragma unroll
        for (int q = 0; q < 4; ++q) an[q] = src[(16 * (t + 1) + q) * step];
      const double *b = tab + ((size_t)t * 64 + lane) * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < NT; ++m)
          acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[(size_t)m * kt * 256 + q], acc[m], 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = an[q];
    }
    // lanes j: 16 consecutive layers of one column
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = 16 * tile + gq + 4 * q;
      if (c >= g.N0) continue;
      double *dst = x + (size_t)c * g.NS + 1;
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        const int k = l0 + 16 * m + j;
        if (k < nzi) dst[k] -= acc[m][q];
      }
    }
  }
}

template <int MT>
static int launch_transform_t(const Geo &g, hipStream_t s, const ModalDev &M, const double *r, double *x,
                              SolverState *st, bool fwd, hipEvent_t *ev) {
  const size_t lds = (size_t)MT * M.kt * 256 * sizeof(double);
  const dim3 grid(M.agrid, M.npanel), blk(MODAL_TB);
  if (fwd && M.batched)
    LAUNCH_TIMED(ev, 0, (k_modal_fwd<MT, true>), grid, blk, lds, s, g, M, r, st);
  else if (fwd)
    LAUNCH_TIMED(ev, 0, (k_modal_fwd<MT, false>), grid, blk, lds, s, g, M, r, st);
  else if (M.batched)
    LAUNCH_TIMED(ev, 0, (k_modal_bwd<MT, true>), grid, blk, lds, s, g, M, x, st);
  else
    LAUNCH_TIMED(ev, 0, (k_modal_bwd<MT, false>), grid, blk, lds, s, g, M, x, st);
  return (int)hipGetLastError();
}

static int launch_transform(const Geo &g, hipStream_t s, const ModalDev &M, const double *r, double *x,
                            SolverState *st, bool fwd, hipEvent_t *ev) {
  switch (M.mt) {
    case 0: return launch_transform_t<0>(g, s, M, r, x, st, fwd, ev);
    case 1: return launch_transform_t<1>(g, s, M, r, x, st, fwd, ev);
    case 2: return launch_transform_t<2>(g, s, M, r, x, st, fwd, ev);
    case 3: return launch_transform_t<3>(g, s, M, r, x, st, fwd, ev);
    case 4: return launch_transform_t<4>(g, s, M, r, x, st, fwd, ev);
    case 5: return launch_transform_t<5>(g, s, M, r, x, st, fwd, ev);
    case 6: return launch_transform_t<6>(g, s, M, r, x, st, fwd, ev);
    case 7: return launch_transform_t<7>(g, s, M, r, x, st, fwd, ev);
    case 8: return launch_transform_t<8>(g, s, M, r, x, st, fwd, ev);
    default: return (int)hipErrorInvalidValue;
  }
}

// --- the 2D solves.  A block owns a mode: FP64 conjugate gradients on
// (L + mu D) x = b, preconditioned by one V-cycle in FP32 (the directions are
// FP32 too; the recurrences for x and the residual are FP64, so the residual
// they carry is x's own).  The V-cycle: a damped Jacobi sweep on the columns
// before and after the coarse correction, a degree-2 Chebyshev polynomial on
// [lmax / 4, lmax] on the levels below (lmax: Gershgorin's bound of the
// mode's D^-1 A), a dense inverse on the coarsest.  The block's only
// synchronisation is its own barrier.  4,096 columns x 48 modes: 0.5 ms for 20
// to 25 iterations, bound by latency (24 cycles a vector memory instruction,
// the vector units 21 % busy).  Four nodes' loads ahead, reciprocals kept
// instead of divisions, and the columns' state in registers gained nothing (the
// last spills).
constexpr int T2 = 1024;  // threads of a 2D block
constexpr int W2 = T2 / 64;

// the block's vectors: in LDS or in the mode's workspace (the same branch
// for every thread)
struct Vec {
  float *g;
  int off;
  bool l;
};

__device__ inline float *lds2d() {
  extern __shared__ __align__(16) unsigned char nsx_dyn_lds[];
  return reinterpret_cast<float *>(nsx_dyn_lds);
}
__device__ inline Vec vec_at(const VecLoc &v, float *work) { return {work + (v.lds ? 0 : v.off), v.off, v.lds != 0}; }
__device__ inline float vget(const Vec &v, int i) { return v.l ? lds2d()[v.off + i] : v.g[i]; }
__device__ inline void vset(const Vec &v, int i, float a) {
  if (v.l)
    lds2d()[v.off + i] = a;
  else
    v.g[i] = a;
}

// sum over row r of a matrix in slices of 64 rows
__device__ inline float sell_row(const SellDev &S, const Vec &v, int r) {
  const int s = __builtin_amdgcn_readfirstlane(r >> 6), e0 = S.ptr[s], e1 = S.ptr[s + 1];
  float a = 0.f;
  if (v.l) {
    const float *x = lds2d() + v.off;
#pragma unroll 4
    for (int e = e0 + (r & 63); e < e1; e += 64) a = fmaf(S.val[e], x[S.col[e]], a);
  } else {
#pragma unroll 4
    for (int e = e0 + (r & 63); e < e1; e += 64) a = fmaf(S.val[e], v.g[S.col[e]], a);
  }
  return a;
}

// sum over the block; one barrier (the two halves of `sh` alternate, so a
// half is rewritten only after every thread has passed the barrier that
// follows its last read)
__device__ inline double block_sum(double v, double (*sh)[W2], int &turn) {
  double a[1] = {v};
  wave_sum<1>(a);
  double *h = sh[turn];
  turn ^= 1;
  if ((threadIdx.x & 63) == 0) h[threadIdx.x >> 6] = a[0];
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < W2; ++w) s += h[w];
  return s;
}

// the V-cycle from level l0 >= 1 down and back up to its solution y, for one
// mode; on entry the level's right-hand side b, its vector t holding the
// first Chebyshev step b / (th d) (l0 not the coarsest), with a barrier since
__device__ inline void cycle_below(const ModalDev &M, int m, float mu, float *work, int l0) {
  const int tid = threadIdx.x, L = M.nlev;
  for (int l = l0; l + 1 < L; ++l) {
    const ModalLevelDev &A = M.lev[l], &C = M.lev[l + 1];
    const Vec b = vec_at(A.b, work), t = vec_at(A.t, work), y = vec_at(A.y, work), bc = vec_at(C.b, work),
              tc = vec_at(C.t, work);
    const Cheb c = A.cheb[m];
    for (int i = tid; i < A.n; i += T2) {
      const float d = fmaf(mu, A.area[i], A.diag[i]), t0 = vget(t, i);
      const float r1 = vget(b, i) - d * t0 - sell_row(A.A, t, i);
      vset(y, i, t0 + c.c1 * t0 + c.c2 * r1 / d);
    }
    __syncthreads();
    for (int i = tid; i < A.n; i += T2) {
      const float d = fmaf(mu, A.area[i], A.diag[i]);
      vset(t, i, vget(b, i) - d * vget(y, i) - sell_row(A.A, y, i));
    }
    __syncthreads();
    const bool last = l + 2 == L;
    const float ith = last ? 0.f : C.cheb[m].ith;
    for (int i = tid; i < C.n; i += T2) {
      const float v = sell_row(A.R, t, i);
      vset(bc, i, v);
      if (!last) vset(tc, i, v * ith / fmaf(mu, C.area[i], C.diag[i]));
    }
    __syncthreads();
  }
  // the coarsest level: eight lanes per row
  {
    const ModalLevelDev &A = M.lev[L - 1];
    const Vec b = vec_at(A.b, work), y = vec_at(A.y, work);
    const float *ci = M.cinv + (size_t)m * M.nc * M.nc;
    for (int i0 = 0; i0 < M.nc; i0 += T2 / 8) {
      const int i = i0 + (tid >> 3);
      float a = 0.f;
      if (i < M.nc)
        for (int k = tid & 7; k < M.nc; k += 8) a = fmaf(ci[(size_t)i * M.nc + k], vget(b, k), a);
      a += __shfl_xor(a, 4, 64);
      a += __shfl_xor(a, 2, 64);
      a += __shfl_xor(a, 1, 64);
      if (i < M.nc && (tid & 7) == 0) vset(y, i, a);
    }
    __syncthreads();
  }
  for (int l = L - 2; l >= l0; --l) {
    const ModalLevelDev &A = M.lev[l];
    const Vec yc = vec_at(M.lev[l + 1].y, work), b = vec_at(A.b, work), t = vec_at(A.t, work), y = vec_at(A.y, work);
    const Cheb c = A.cheb[m];
    for (int i = tid; i < A.n; i += T2) vset(y, i, vget(y, i) + sell_row(A.P, yc, i));
    __syncthreads();
    for (int i = tid; i < A.n; i += T2) {
      const float d = fmaf(mu, A.area[i], A.diag[i]);
      const float r2 = vget(b, i) - d * vget(y, i) - sell_row(A.A, y, i);
      vset(b, i, r2);
      vset(t, i, r2 * c.ith / d);
    }
    __syncthreads();
    for (int i = tid; i < A.n; i += T2) {
      const float d = fmaf(mu, A.area[i], A.diag[i]), t0 = vget(t, i);
      const float r3 = vget(b, i) - d * t0 - sell_row(A.A, t, i);
      vset(y, i, vget(y, i) + t0 + c.c1 * t0 + c.c2 * r3 / d);
    }
    __syncthreads();
  }
}

struct V3 {
  int a, b, c;
};

__global__ __launch_bounds__(T2) void k_modal_2d(ModalDev M, SolverState *st) {
  if (st->done) return;
  __shared__ double sh[2][W2];
  int turn = 0;
  const int m = blockIdx.x, tid = threadIdx.x, N0 = M.N0, L = M.nlev;
  const double mu64 = M.mu[m];
  const float mu = (float)mu64, om = NSX_MODAL_OMEGA;
  double *r = M.bh + (size_t)m * M.N0p, *x = M.xh + (size_t)m * M.N0p, *ap = M.ap + (size_t)m * M.N0p;
  float *work = M.work + (size_t)m * M.nwork;
  const V3 *nb = reinterpret_cast<const V3 *>(M.nb);

  // the modes share the square of the residual's target evenly
  double part = 0.0;
  for (int q = tid; q < M.agrid * M.npanel; q += T2) part += M.part[q];
  const double total = block_sum(part, sh, turn);
  if (m == 0) {
    // the mode's null space is the constants: the mean that rounding leaves in
    // its right-hand side is no part of the problem
    double s = 0.0;
    for (int i = tid; i < N0; i += T2) s += r[i];
    const double mean = block_sum(s, sh, turn) / N0;
    for (int i = tid; i < N0; i += T2) r[i] -= mean;
  }
  double own = 0.0;
  for (int i = tid; i < N0; i += T2) own += r[i] * r[i];
  const double r0 = block_sum(own, sh, turn);
  const double target = st->m_tau * st->m_tau * total / M.nzi;
  if (!(r0 > target) || !isfinite(r0)) {
    for (int i = tid; i < N0; i += T2) x[i] = 0.0;
    return;
  }
  const double scale = sqrt(r0), inv = 1.0 / scale;

  const Vec V = vec_at(M.lev[0].y, work), Z = vec_at(M.z0, work);
  Vec P0 = vec_at(M.p[0], work), P1 = vec_at(M.p[1], work);
  const float *dg = M.lev[0].diag, *ar = M.lev[0].area;
  for (int i = tid; i < N0; i += T2) {
    x[i] = 0.0;
    vset(V, i, om * (float)(r[i] * inv) / fmaf(mu, ar[i], dg[i]));
  }
  __syncthreads();

  double rho_old = 1.0, rr = r0;
  int it = 0;
  while (rr > target && it < 100) {
    // z = M^-1 r / scale
    if (L == 1) {
      // the columns are the coarsest level
      const float *ci = M.cinv + (size_t)m * M.nc * M.nc;
      for (int i = tid; i < N0; i += T2) vset(P1, i, (float)(r[i] * inv));
      __syncthreads();
      for (int i = tid; i < N0; i += T2) {
        float a = 0.f;
        for (int k = 0; k < N0; ++k) a = fmaf(ci[(size_t)i * M.nc + k], vget(P1, k), a);
        vset(Z, i, a);
      }
    } else {
      // the columns: residual of the first sweep (V = omega r / d)
      for (int i = tid; i < N0; i += T2) {
        const V3 n = nb[i];
        const float4 w = M.wa[i];
        const float v = vget(V, i), d = fmaf(mu, w.w, w.x + w.y + w.z);
        float a = (float)(r[i] * inv) - d * v;
        if (V.l) {
          const float *q = lds2d() + V.off;
          a = fmaf(w.x, q[n.a], fmaf(w.y, q[n.b], fmaf(w.z, q[n.c], a)));
        } else {
          a = fmaf(w.x, V.g[n.a], fmaf(w.y, V.g[n.b], fmaf(w.z, V.g[n.c], a)));
        }
        vset(Z, i, a);
      }
      __syncthreads();
      {
        const ModalLevelDev &C = M.lev[1];
        const Vec bc = vec_at(C.b, work), tc = vec_at(C.t, work);
        const float ith = L == 2 ? 0.f : C.cheb[m].ith;
        for (int i = tid; i < C.n; i += T2) {
          const float v = sell_row(M.lev[0].R, Z, i);
          vset(bc, i, v);
          if (L > 2) vset(tc, i, v * ith / fmaf(mu, C.area[i], C.diag[i]));
        }
        __syncthreads();
      }
      cycle_below(M, m, mu, work, 1);
      {
        const Vec y1 = vec_at(M.lev[1].y, work);
        for (int i = tid; i < N0; i += T2) vset(V, i, vget(V, i) + sell_row(M.lev[0].P, y1, i));
        __syncthreads();
      }
    }
    // the columns' second sweep and rho = <r, z>
    double acc = 0.0;
    for (int i = tid; i < N0; i += T2) {
      const float rs = (float)(r[i] * inv);
      float z;
      if (L == 1) {
        z = vget(Z, i);
      } else {
        const V3 n = nb[i];
        const float4 w = M.wa[i];
        const float v = vget(V, i), d = fmaf(mu, w.w, w.x + w.y + w.z);
        float a = fmaf(-d, v, rs);
        if (V.l) {
          const float *q = lds2d() + V.off;
          a = fmaf(w.x, q[n.a], fmaf(w.y, q[n.b], fmaf(w.z, q[n.c], a)));
        } else {
          a = fmaf(w.x, V.g[n.a], fmaf(w.y, V.g[n.b], fmaf(w.z, V.g[n.c], a)));
        }
        z = v + om * a / d;
        vset(Z, i, z);
      }
      acc += (r[i] * inv) * (double)z;
    }
    const double rho = block_sum(acc, sh, turn);
    const float beta = it == 0 ? 0.f : (float)(rho / rho_old);
    rho_old = rho;
    // p = z + beta p and A p in FP64
    acc = 0.0;
    for (int i = tid; i < N0; i += T2) {
      const V3 n = nb[i];
      const double *w = M.w64 + 3 * (size_t)i;
      const double w0 = w[0], w1 = w[1], w2 = w[2];
      float p[4];
      const int id[4] = {i, n.a, n.b, n.c};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        p[q] = vget(Z, id[q]);
        if (it > 0) p[q] = fmaf(beta, vget(P0, id[q]), p[q]);
      }
      const double pd = (double)p[0];
      const double a = w0 * (pd - (double)p[1]) + w1 * (pd - (double)p[2]) + w2 * (pd - (double)p[3]) +
                       mu64 * M.area64[i] * pd;
      vset(P1, i, p[0]);
      ap[i] = a;
      acc += pd * a;
    }
    const double pap = block_sum(acc, sh, turn);
    const double alpha = rho / pap;
    if (!(pap > 0.0) || !isfinite(alpha)) break;
    // x, r and the next first sweep
    const double as = alpha * scale;
    acc = 0.0;
    for (int i = tid; i < N0; i += T2) {
      x[i] += as * (double)vget(P1, i);
      const double rn = r[i] - as * ap[i];
      r[i] = rn;
      acc += rn * rn;
      vset(V, i, om * (float)(rn * inv) / fmaf(mu, ar[i], dg[i]));
    }
    rr = block_sum(acc, sh, turn);
    const Vec sw = P0;
    P0 = P1;
    P1 = sw;
    ++it;
  }
  // no correction from a solve that gained nothing
  if (!(rr < r0))
    for (int i = tid; i < N0; i += T2) x[i] = 0.0;
  if (tid == 0) {
    atomicMax(&st->m_cyc, it);
    atomicAdd(&st->m_swept, it);
  }
}

// --- the 2D solves batched over the modes, for meshes whose vectors pass the
// LDS.  The same CG and V-cycle on node-major arrays (rows of mp modes), one
// launch per sweep over the chip: a thread holds four modes of a node, so the
// graph's indices and weights are read once for all modes (one block per mode
// reads them per mode, and is bound by its CU's address unit: 500 us an
// iteration at 65,536 columns x 96 layers, against about 300 on average here).  The columns' smoother is
// the Chebyshev one too, on the mode's own bounds: the high modes, most of the
// work, take 6 to 11 iterations for 1e-10 instead of 11 to 17, for two more sweeps.
// Levels 2 and below run one block per mode in LDS.  Modes whose residual has
// met its target stop; the rows are swept up to the last mode still
// iterating.  At 6.3M prisms with all modes iterating the update moves 350 MB
// in 75 us (4.6 TB/s) and the product 126 MB and its gathers in 46 us.  On
// average 34 modes are swept, at 1.09 TB/s of the columns' vectors: 18 kernels of
// 5 to 40 us, a tenth of the time between them.
constexpr int MB = NSX_BLOCK;

// f(node, q, K) over the nodes and the groups q of four modes below nact; a
// thread keeps its q, so what depends on the modes alone (K = make(q)) is
// read once; blocks take contiguous runs of nodes, an XCD's blocks adjacent
// ones
template <class K, class F>
__device__ inline void mb_nodes(int n, int nact, K &&make, F &&f) {
  const int n4 = (nact + 3) >> 2, nper = MB / n4, q = threadIdx.x % n4, row = threadIdx.x / n4;
  const int ng = (n + nper - 1) / nper, G = gridDim.x, b = blockIdx.x;
  const int lb = (G % NSX_NXCD) == 0 ? (b % NSX_NXCD) * (G / NSX_NXCD) + b / NSX_NXCD : b;
  const int per = (ng + G - 1) / G, g0 = lb * per, g1 = g0 + per < ng ? g0 + per : ng;
  if (row >= nper || g0 >= g1) return;
  const auto k = make(q);
  for (int g = g0; g < g1; ++g) {
    const int i = g * nper + row;
    if (i < n) f(i, q, k);
  }
}

struct F4 {
  float v[4];
};
__device__ inline F4 ldf(const float *p) {
  const float4 a = *(const float4 *)p;
  return {{a.x, a.y, a.z, a.w}};
}
__device__ inline void stf(float *p, const F4 &a) { *(float4 *)p = make_float4(a.v[0], a.v[1], a.v[2], a.v[3]); }

// sum over row i of a CSR matrix times the node-major x
__device__ inline F4 csr_row(const CsrDev &A, const float *x, int mp, int i, int q) {
  F4 s = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 2
  for (int e = A.ptr[i]; e < A.ptr[i + 1]; ++e) {
    const float w = A.val[e];
    const F4 a = ldf(x + (size_t)A.col[e] * mp + 4 * q);
#pragma unroll
    for (int k = 0; k < 4; ++k) s.v[k] = fmaf(w, a.v[k], s.v[k]);
  }
  return s;
}

// per-mode sums of a block: thread (row, q) adds acc to mode 4 q + k; row by
// row in order, so the sums are the same in every run
__device__ inline void mb_partials(const ModalDev &M, double *P, const double (&acc)[4], int nact) {
  __shared__ double sh[MB][4];
  const int n4 = (nact + 3) >> 2, nper = MB / n4;
#pragma unroll
  for (int k = 0; k < 4; ++k) sh[threadIdx.x][k] = acc[k];
  __syncthreads();
  for (int m = threadIdx.x; m < 4 * n4; m += MB) {
    double s = 0.0;
    for (int r = 0; r < nper; ++r) s += sh[r * n4 + (m >> 2)][m & 3];
    P[(size_t)blockIdx.x * M.mp + m] = s;
  }
}

// the sum of mode 0 (its null space is the constants: the mean that rounding
// leaves in it is no part of the problem)
__global__ __launch_bounds__(MB) void k_mb_mean(ModalDev M, const SolverState *st) {
  if (st->done) return;
  double s[1] = {0.0};
  for (int i = blockIdx.x * MB + threadIdx.x; i < M.N0; i += gridDim.x * MB) s[0] += M.bh[(size_t)i * M.mp];
  write_partials<1>(s, M.rpart);
}

// |r_m|^2 of every mode, mode 0 without its mean
__global__ __launch_bounds__(MB) void k_mb_norm(ModalDev M, const SolverState *st) {
  if (st->done) return;
  double mean[1];
  reduce_partials<1>(M.rpart, NSX_MB_MEAN, mean);
  __syncthreads();
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const double m0 = mean[0] / M.N0;
  mb_nodes(M.N0, M.mp, [](int) { return 0; }, [&](int i, int q, int) {
    double r[4];
    double *p = M.bh + (size_t)i * M.mp + 4 * q;
    ld4(p, r);
    if (q == 0) {
      r[0] -= m0;
      p[0] = r[0];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] += r[k] * r[k];
  });
  mb_partials(M, M.rpart2, acc, M.mp);
}

// The scalars of 16 modes per block from the partial sums of the kernel
// before.  WHAT 0: the start (targets, scales); 1: rho and beta; 2: alpha;
// 3: |r|^2 and which modes go on (nact of iteration it + 1)
template <int WHAT>
__global__ __launch_bounds__(T2) void k_mb_scalars(ModalDev M, SolverState *st, int it) {
  if (st->done) return;
  const int cur = WHAT == 0 ? M.mp : M.nact[it];
  if (cur == 0) return;
  // 64 slices of the rows, 16 modes each
  __shared__ double sh[T2 / 16][17], shw[2][W2];
  const int j = threadIdx.x & 15, sl = threadIdx.x >> 4, m = 16 * (int)blockIdx.x + j;
  double s = 0.0;
  if (m < cur)
#pragma unroll 8
    for (int b = sl; b < NSX_MB_GRID; b += T2 / 16) s += M.rpart2[(size_t)b * M.mp + m];
  sh[sl][j] = s;
  double total = 0.0;
  if (WHAT == 0) {
    int turn = 0;
    double tp = 0.0;
    for (int q = threadIdx.x; q < M.agrid * M.npanel; q += T2) tp += M.part[q];
    total = block_sum(tp, shw, turn);
  } else {
    __syncthreads();
  }
  if (sl != 0 || m >= cur) return;
  s = 0.0;
  for (int w = 0; w < T2 / 16; ++w) s += sh[w][j];
  ModeState &S = M.ms[m];
  if (WHAT == 0) {
    const double target = st->m_tau * st->m_tau * total / M.nzi;
    S.rr = S.r0 = s;
    S.target = target;
    S.act = s > target && isfinite(s);
    S.scale = S.act ? sqrt(s) : 1.0;
    S.inv = 1.0 / S.scale;
    S.as = 0.0;
    S.beta = 0.f;
    if (S.act) atomicMax(&M.nact[0], m + 1);
  } else if (WHAT == 1) {
    S.beta = S.act && it > 0 ? (float)(s / S.rho) : 0.f;
    S.rho = s;
  } else if (WHAT == 2) {
    const double alpha = S.rho / s;
    if (S.act && !(s > 0.0 && isfinite(alpha))) S.act = 0;
    S.as = S.act ? alpha * S.scale : 0.0;
  } else {
    S.rr = s;
    S.act = S.act && s > S.target;
    if (S.act) {
      atomicMax(&M.nact[it + 1], m + 1);
    } else {
      // the sweeps go on over its group of four, and these scalars are not
      // formed again past the last mode still iterating: no further step
      S.as = 0.0;
      S.beta = 0.f;
    }
    if (m == 0) {
      st->m_cyc = it + 1;
      st->m_swept += cur;
    }
  }
}

__global__ void k_mb_clear(ModalDev M, const SolverState *st) {
  if (st->done) return;
  for (int q = threadIdx.x; q <= NSX_MB_ITERS; q += blockDim.x) M.nact[q] = 0;
}

struct FourCheb {
  float mu[4];
  Cheb c[4];
};
__device__ inline FourCheb four_cheb(const ModalDev &M, const ModalLevelDev &A, int q) {
  FourCheb k;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    k.mu[c] = (float)M.mu[4 * q + c];
    k.c[c] = A.cheb[4 * q + c];
  }
  return k;
}

// x += alpha p, r -= alpha A p, |r|^2, the V-cycle's right-hand side R = r /
// scale and its first Chebyshev step V = R / (th d) (first: x = 0 and those)
template <bool FIRST>
__global__ __launch_bounds__(MB) void k_mb_update(ModalDev M, const float *p, const SolverState *st, int it) {
  if (st->done) return;
  const int nact = M.nact[it], mp = M.mp;
  if (!FIRST && nact == 0) return;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const float *dg = M.lev[0].diag, *ar = M.lev[0].area;
  struct Kon {
    float mu[4], ith[4];
    double inv[4], as[4];
  };
  auto make = [&](int q) {
    Kon k;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      k.mu[c] = (float)M.mu[4 * q + c];
      k.ith[c] = M.lev[0].cheb[4 * q + c].ith;
      k.inv[c] = M.ms[4 * q + c].inv;
      k.as[c] = M.ms[4 * q + c].as;
    }
    return k;
  };
  mb_nodes(M.N0, FIRST ? mp : nact, make, [&](int i, int q, const Kon &K) {
    const size_t s = (size_t)i * mp + 4 * q;
    double r[4], x[4] = {0.0, 0.0, 0.0, 0.0};
    ld4(M.bh + s, r);
    if (!FIRST) {
      double a[4];
      ld4(M.xh + s, x);
      ld4(M.ap + s, a);
      const F4 pv = ldf(p + s);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        x[k] += K.as[k] * (double)pv.v[k];
        r[k] -= K.as[k] * a[k];
        acc[k] += r[k] * r[k];
      }
      st4(M.bh + s, r);
    }
    st4(M.xh + s, x);
    const float d0 = dg[i], a0 = ar[i];
    F4 rs, v;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      rs.v[k] = (float)(r[k] * K.inv[k]);
      v.v[k] = rs.v[k] * K.ith[k] / fmaf(K.mu[k], a0, d0);
    }
    stf(M.R + s, rs);
    stf(M.V + s, v);
  });
  if (!FIRST) mb_partials(M, M.rpart2, acc, nact);
}

// the columns' sweeps, as k_mb_smooth's on level 1.  WHAT 0: Z = the Chebyshev
// sweep from zero (V holds its first step); 1: V = R - A Z; 2: W = R - A Z, V
// = the first step on it; 3: z = Z + the sweep's rest, partial <r, z>
template <int WHAT>
__global__ __launch_bounds__(MB) void k_mb_columns(ModalDev M, const SolverState *st, int it) {
  if (st->done) return;
  const int nact = M.nact[it], mp = M.mp;
  if (nact == 0) return;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  auto make = [&](int q) { return four_cheb(M, M.lev[0], q); };
  mb_nodes(M.N0, nact, make, [&](int i, int q, const FourCheb &K) {
    const size_t s = (size_t)i * mp + 4 * q;
    constexpr bool ON_V = WHAT == 0 || WHAT == 3;  // A applied to V, else to Z
    const float *src = ON_V ? M.V : M.Z;
    const V3 n = reinterpret_cast<const V3 *>(M.nb)[i];
    const float4 w = M.wa[i];
    const F4 c = ldf(src + s), a0 = ldf(src + (size_t)n.a * mp + 4 * q), a1 = ldf(src + (size_t)n.b * mp + 4 * q),
             a2 = ldf(src + (size_t)n.c * mp + 4 * q), b = ldf((WHAT == 3 ? M.W : M.R) + s);
    F4 z, rr, o, o2;
    if (WHAT == 3) {
      z = ldf(M.Z + s);
      rr = ldf(M.R + s);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float d = fmaf(K.mu[k], w.w, w.x + w.y + w.z);
      const float r = fmaf(w.x, a0.v[k], fmaf(w.y, a1.v[k], fmaf(w.z, a2.v[k], fmaf(-d, c.v[k], b.v[k]))));
      o.v[k] = r;
      if (ON_V) o.v[k] = (WHAT == 3 ? z.v[k] : 0.f) + c.v[k] + K.c[k].c1 * c.v[k] + K.c[k].c2 * r / d;
      if (WHAT == 2) o2.v[k] = r * K.c[k].ith / d;
      if (WHAT == 3) acc[k] += (double)rr.v[k] * (double)o.v[k];
    }
    stf((ON_V ? M.Z : WHAT == 1 ? M.V : M.W) + s, o);
    if (WHAT == 2) stf(M.V + s, o2);
  });
  if (WHAT == 3) mb_partials(M, M.rpart2, acc, nact);
}

// p = z + beta p_old at the column and its neighbours, A p in FP64, <p, A p>
__global__ __launch_bounds__(MB) void k_mb_ap(ModalDev M, const float *pold, float *pnew, const SolverState *st,
                                              int it) {
  if (st->done) return;
  const int nact = M.nact[it], mp = M.mp;
  if (nact == 0) return;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  struct Kon {
    float beta[4];
    double mu[4];
  };
  auto make = [&](int q) {
    Kon k;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      k.beta[c] = M.ms[4 * q + c].beta;
      k.mu[c] = M.mu[4 * q + c];
    }
    return k;
  };
  mb_nodes(M.N0, nact, make, [&](int i, int q, const Kon &K) {
    const V3 n = reinterpret_cast<const V3 *>(M.nb)[i];
    const double *w = M.w64 + 3 * (size_t)i;
    const int id[4] = {i, n.a, n.b, n.c};
    F4 p[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const size_t s = (size_t)id[c] * mp + 4 * q;
      p[c] = ldf(M.Z + s);
      if (it > 0) {
        const F4 o = ldf(pold + s);
#pragma unroll
        for (int k = 0; k < 4; ++k) p[c].v[k] = fmaf(K.beta[k], o.v[k], p[c].v[k]);
      }
    }
    const double w0 = w[0], w1 = w[1], w2 = w[2], ar = M.area64[i];
    double a[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double pd = (double)p[0].v[k];
      a[k] = w0 * (pd - (double)p[1].v[k]) + w1 * (pd - (double)p[2].v[k]) + w2 * (pd - (double)p[3].v[k]) +
             K.mu[k] * ar * pd;
      acc[k] += pd * a[k];
    }
    const size_t s = (size_t)i * mp + 4 * q;
    stf(pnew + s, p[0]);
    st4(M.ap + s, a);
  });
  mb_partials(M, M.rpart2, acc, nact);
}

// b of the level below = R src, and (t not null) its first Chebyshev step
__global__ __launch_bounds__(MB) void k_mb_restrict(ModalDev M, CsrDev R, int lc, const float *src, float *b, float *t,
                                                    const SolverState *st, int it) {
  if (st->done) return;
  const int nact = M.nact[it], mp = M.mp;
  if (nact == 0) return;
  const ModalLevelDev &C = M.lev[lc];
  struct Kon {
    float mu[4], ith[4];
  };
  auto make = [&](int q) {
    Kon k;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      k.mu[c] = (float)M.mu[4 * q + c];
      k.ith[c] = t ? C.cheb[4 * q + c].ith : 0.f;
    }
    return k;
  };
  mb_nodes(C.n, nact, make, [&](int i, int q, const Kon &K) {
    const size_t s = (size_t)i * mp + 4 * q;
    const F4 v = csr_row(R, src, mp, i, q);
    stf(b + s, v);
    if (t) {
      const float dg = C.diag[i], ar = C.area[i];
      F4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) o.v[k] = v.v[k] * K.ith[k] / fmaf(K.mu[k], ar, dg);
      stf(t + s, o);
    }
  });
}

__global__ __launch_bounds__(MB) void k_mb_prolong(ModalDev M, CsrDev P, int n, const float *yc, float *y,
                                                   const SolverState *st, int it) {
  if (st->done) return;
  const int nact = M.nact[it], mp = M.mp;
  if (nact == 0) return;
  mb_nodes(n, nact, [](int) { return 0; }, [&](int i, int q, int) {
    const size_t s = (size_t)i * mp + 4 * q;
    const F4 a = csr_row(P, yc, mp, i, q);
    F4 v = ldf(y + s);
#pragma unroll
    for (int k = 0; k < 4; ++k) v.v[k] += a.v[k];
    stf(y + s, v);
  });
}

// level 1's sweeps.  WHAT 0: y = the Chebyshev sweep from zero (t holds its
// first step); 1: t = b - A y; 2: b = b - A y, t = the first step on it;
// 3: y += the sweep's rest
template <int WHAT>
__global__ __launch_bounds__(MB) void k_mb_smooth(ModalDev M, const SolverState *st, int it) {
  if (st->done) return;
  const int nact = M.nact[it], mp = M.mp;
  if (nact == 0) return;
  const ModalLevelDev &A = M.lev[1];
  auto make = [&](int q) { return four_cheb(M, A, q); };
  mb_nodes(A.n, nact, make, [&](int i, int q, const FourCheb &K) {
    const size_t s = (size_t)i * mp + 4 * q;
    constexpr bool ON_T = WHAT == 0 || WHAT == 3;  // A applied to t, else to y
    const float *src = ON_T ? M.t1 : M.y1;
    const F4 a = csr_row(A.Ac, src, mp, i, q), c = ldf(src + s), b = ldf(M.b1 + s);
    const float dg = A.diag[i], ar = A.area[i];
    F4 y, o, o2;
    if (WHAT == 3) y = ldf(M.y1 + s);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const Cheb h = K.c[k];
      const float d = fmaf(K.mu[k], ar, dg), r = b.v[k] - d * c.v[k] - a.v[k];
      o.v[k] = r;
      if (ON_T) o.v[k] = (WHAT == 3 ? y.v[k] : 0.f) + c.v[k] + h.c1 * c.v[k] + h.c2 * r / d;
      if (WHAT == 2) o2.v[k] = r * h.ith / d;
    }
    stf((ON_T ? M.y1 : WHAT == 1 ? M.t1 : M.b1) + s, o);
    if (WHAT == 2) stf(M.t1 + s, o2);
  });
}

// levels 2 and below, a block per mode
__global__ __launch_bounds__(T2) void k_mb_below(ModalDev M, const SolverState *st, int it) {
  if (st->done) return;
  const int m = blockIdx.x, mp = M.mp, tid = threadIdx.x;
  if (m >= M.nact[it] || !M.ms[m].act) return;
  const ModalLevelDev &A = M.lev[2];
  float *work = M.work + (size_t)m * M.nwork;
  const float mu = (float)M.mu[m];
  const Vec b = vec_at(A.b, work), t = vec_at(A.t, work), y = vec_at(A.y, work);
  const bool last = M.nlev == 3;
  const float ith = last ? 0.f : A.cheb[m].ith;
  for (int i = tid; i < A.n; i += T2) {
    const float v = M.b2[(size_t)i * mp + m];
    vset(b, i, v);
    if (!last) vset(t, i, v * ith / fmaf(mu, A.area[i], A.diag[i]));
  }
  __syncthreads();
  cycle_below(M, m, mu, work, 2);
  for (int i = tid; i < A.n; i += T2) M.y2[(size_t)i * mp + m] = vget(y, i);
}

// the queue's end after `it` iterations: wait for more, or the cycle's end (no
// correction from a mode whose solve gained nothing)
__global__ __launch_bounds__(MB) void k_mb_final(ModalDev M, SolverState *st, int it) {
  if (st->done) return;
  if (it < NSX_MB_ITERS && M.nact[it] > 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->m_wait = it;
      st->done = NSX_WAITS;
    }
    return;
  }
  bool any = false;
  for (int m = 0; m < M.nzi; ++m) any = any || !(M.ms[m].rr <= M.ms[m].r0);
  if (!any) return;
  for (size_t s = (size_t)blockIdx.x * MB + threadIdx.x; s < (size_t)M.N0 * M.mp; s += (size_t)gridDim.x * MB) {
    const ModeState &S = M.ms[s % M.mp];
    if (!(S.rr <= S.r0)) M.xh[s] = 0.0;
  }
}

__global__ void k_modal_resume(SolverState *st) {
  if (st->done == NSX_WAITS) st->done = 0;
}

static int launch_batched(hipStream_t s, const ModalDev &M, SolverState *st, int it0, int iters) {
  const dim3 grid(NSX_MB_GRID), blk(MB), sc(M.kt);
  if (it0 == 0) {
    hipLaunchKernelGGL(k_mb_clear, dim3(1), dim3(64), 0, s, M, st);
    hipLaunchKernelGGL(k_mb_mean, dim3(NSX_MB_MEAN), blk, 0, s, M, st);
    hipLaunchKernelGGL(k_mb_norm, grid, blk, 0, s, M, st);
    hipLaunchKernelGGL(k_mb_scalars<0>, sc, dim3(T2), 0, s, M, st, 0);
    hipLaunchKernelGGL(k_mb_update<true>, grid, blk, 0, s, M, (const float *)nullptr, st, 0);
  }
  const ModalLevelDev &C = M.lev[0], &A = M.lev[1];
  const int end = it0 + iters < NSX_MB_ITERS ? it0 + iters : NSX_MB_ITERS;
  for (int it = it0; it < end; ++it) {
    hipLaunchKernelGGL(k_mb_columns<0>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_columns<1>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_restrict, grid, blk, 0, s, M, C.Rc, 1, (const float *)M.V, M.b1, M.t1, st, it);
    hipLaunchKernelGGL(k_mb_smooth<0>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_smooth<1>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_restrict, grid, blk, 0, s, M, A.Rc, 2, (const float *)M.t1, M.b2, (float *)nullptr, st, it);
    hipLaunchKernelGGL(k_mb_below, dim3(M.nzi), dim3(T2), (size_t)M.lds2d, s, M, st, it);
    hipLaunchKernelGGL(k_mb_prolong, grid, blk, 0, s, M, A.Pc, A.n, (const float *)M.y2, M.y1, st, it);
    hipLaunchKernelGGL(k_mb_smooth<2>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_smooth<3>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_prolong, grid, blk, 0, s, M, C.Pc, M.N0, (const float *)M.y1, M.Z, st, it);
    hipLaunchKernelGGL(k_mb_columns<2>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_columns<3>, grid, blk, 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_scalars<1>, sc, dim3(T2), 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_ap, grid, blk, 0, s, M, (const float *)M.P[it & 1], M.P[(it + 1) & 1], st, it);
    hipLaunchKernelGGL(k_mb_scalars<2>, sc, dim3(T2), 0, s, M, st, it);
    hipLaunchKernelGGL(k_mb_update<false>, grid, blk, 0, s, M, (const float *)M.P[(it + 1) & 1], st, it);
    hipLaunchKernelGGL(k_mb_scalars<3>, sc, dim3(T2), 0, s, M, st, it);
  }
  hipLaunchKernelGGL(k_mb_final, grid, blk, 0, s, M, st, end);
  return (int)hipGetLastError();
}

int launch_modal_resume(hipStream_t s, SolverState *st) {
  hipLaunchKernelGGL(k_modal_resume, dim3(1), dim3(1), 0, s, st);
  return (int)hipGetLastError();
}

int launch_modal_fwd(const Geo &g, hipStream_t s, const ModalDev &M, const double *r, SolverState *st,
                     hipEvent_t *ev) {
  return launch_transform(g, s, M, r, nullptr, st, true, ev);
}

int launch_modal_2d(hipStream_t s, const ModalDev &M, SolverState *st, int it0, int iters, hipEvent_t *ev) {
  if (M.batched) {
    if (ev) (void)hipEventRecord(ev[0], s);
    const int rc = launch_batched(s, M, st, it0, iters);
    if (ev) (void)hipEventRecord(ev[1], s);
    return rc;
  }
  LAUNCH_TIMED(ev, 0, k_modal_2d, dim3(M.nzi), dim3(T2), (size_t)M.lds2d, s, M, st);
  return (int)hipGetLastError();
}

int launch_modal_bwd(const Geo &g, hipStream_t s, const ModalDev &M, double *x, SolverState *st, hipEvent_t *ev) {
  return launch_transform(g, s, M, nullptr, x, st, false, ev);
}

static bool allow(const void *kern, int lds) {
  return hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
}

template <int MT>
static bool allow_t(int lds) {
  return allow(reinterpret_cast<const void *>(&k_modal_fwd<MT, false>), lds) &&
         allow(reinterpret_cast<const void *>(&k_modal_fwd<MT, true>), lds) &&
         allow(reinterpret_cast<const void *>(&k_modal_bwd<MT, false>), lds) &&
         allow(reinterpret_cast<const void *>(&k_modal_bwd<MT, true>), lds);
}

// raises the kernels' dynamic LDS limits to what M asks for
bool modal_allow_lds(const ModalDev &M) {
  const int tr = M.mt * M.kt * 256 * (int)sizeof(double);
  const bool ok = M.batched ? allow(reinterpret_cast<const void *>(&k_mb_below), M.lds2d)
                            : allow(reinterpret_cast<const void *>(&k_modal_2d), M.lds2d);
  switch (M.mt) {
    case 0: return ok;
    case 1: return ok && allow_t<1>(tr);
    case 2: return ok && allow_t<2>(tr);
    case 3: return ok && allow_t<3>(tr);
    case 4: return ok && allow_t<4>(tr);
    case 5: return ok && allow_t<5>(tr);
    case 6: return ok && allow_t<6>(tr);
    case 7: return ok && allow_t<7>(tr);
    case 8: return ok && allow_t<8>(tr);
    default: return false;
  }
}
