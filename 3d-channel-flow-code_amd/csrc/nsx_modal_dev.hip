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
// passes the LDS).
constexpr int MODAL_TB = 256;

template <int MT>
__device__ inline const double *lds_panel(const double *src, int kt) {
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

template <int MT>
__global__ __launch_bounds__(MODAL_TB) void k_modal_fwd(Geo g, ModalDev M, const double *r, const SolverState *st) {
  if (st->done) return;
  const int kt = M.kt, nzi = M.nzi, m0 = 16 * MT * (int)blockIdx.y;
  const double *tab = lds_panel<MT>(M.tfwd + (size_t)blockIdx.y * MT * kt * 256, kt);
  const int lane = threadIdx.x & 63, j = lane & 15, gq = lane >> 4;
  const int ntile = M.N0p >> 4, stride = gridDim.x * (MODAL_TB / 64);
  double sum[1] = {0.0};
  for (int tile = blockIdx.x * (MODAL_TB / 64) + (threadIdx.x >> 6); tile < ntile; tile += stride) {
    const int c = 16 * tile + j;
    const bool ok = c < g.N0;
    const double *src = r + (size_t)(ok ? c : 0) * g.NS + 1;
    f64x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
    double b[4], bn[4];
    load_layers(src, 4 * gq, nzi, ok, b);
    for (int t = 0; t < kt; ++t) {
      if (t + 1 < kt) load_layers(src, 16 * (t + 1) + 4 * gq, nzi, ok, bn);
      const double *a = tab + ((size_t)t * 64 + lane) * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[(size_t)m * kt * 256 + q], b[q], acc[m], 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) b[q] = bn[q];
    }
    // lanes j: 16 consecutive columns of one mode, a 128-byte run
#pragma unroll
    for (int m = 0; m < MT; ++m)
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

template <int MT>
__global__ __launch_bounds__(MODAL_TB) void k_modal_bwd(Geo g, ModalDev M, double *x, SolverState *st) {
  if (st->done) return;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    st->m_iters += st->m_cyc;
    st->m_cyc = 0;
    st->mp_pass += 1;
  }
  const int kt = M.kt, nzi = M.nzi, l0 = 16 * MT * (int)blockIdx.y;
  const double *tab = lds_panel<MT>(M.tbwd + (size_t)blockIdx.y * MT * kt * 256, kt);
  const int lane = threadIdx.x & 63, j = lane & 15, gq = lane >> 4;
  const int ntile = M.N0p >> 4, stride = gridDim.x * (MODAL_TB / 64);
  for (int tile = blockIdx.x * (MODAL_TB / 64) + (threadIdx.x >> 6); tile < ntile; tile += stride) {
    f64x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
    // xh's padding modes and columns are zero
    const double *src = M.xh + (size_t)(4 * gq) * M.N0p + 16 * tile + j;
    double a[4], an[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = src[(size_t)q * M.N0p];
    for (int t = 0; t < kt; ++t) {
      if (t + 1 < kt)
#pragma unroll
        for (int q = 0; q < 4; ++q) an[q] = src[(size_t)(16 * (t + 1) + q) * M.N0p];
      const double *b = tab + ((size_t)t * 64 + lane) * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < MT; ++m)
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
      for (int m = 0; m < MT; ++m) {
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
  if (fwd)
    LAUNCH_TIMED(ev, 0, k_modal_fwd<MT>, grid, blk, lds, s, g, M, r, st);
  else
    LAUNCH_TIMED(ev, 0, k_modal_bwd<MT>, grid, blk, lds, s, g, M, x, st);
  return (int)hipGetLastError();
}

static int launch_transform(const Geo &g, hipStream_t s, const ModalDev &M, const double *r, double *x,
                            SolverState *st, bool fwd, hipEvent_t *ev) {
  switch (M.mt) {
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
// synchronisation is its own barrier.
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

// Chebyshev steps of degree 2 on [lmax/4, lmax]: first = r / (th d), then
// c1 first + c2 r' / d
struct Cheb {
  float ith, c1, c2;
};
__device__ inline Cheb cheb_of(float lmax) {
  const float th = 0.625f * lmax, de = 0.375f * lmax, rho0 = de / th, rho1 = 1.f / (2.f * th / de - rho0);
  return {1.f / th, rho1 * rho0, 2.f * rho1 / de};
}

struct Lvl {
  Vec y, t, b;
  Cheb c;
};

struct V3 {
  int a, b, c;
};

__global__ __launch_bounds__(T2) void k_modal_2d(ModalDev M, SolverState *st) {
  if (st->done) return;
  __shared__ double sh[2][W2];
  __shared__ Cheb cheb[NSX_MODAL_MAXLEV];
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

  // this mode's Gershgorin bounds on the levels between
  __syncthreads();
  for (int l = 1; l + 1 < L; ++l) {
    const ModalLevelDev &A = M.lev[l];
    float b = 1.f;
    for (int i = tid; i < A.n; i += T2) b = fmaxf(b, 1.f + A.sabs[i] / fmaf(mu, A.area[i], A.diag[i]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) b = fmaxf(b, __shfl_xor(b, o, 64));
    __syncthreads();
    if ((tid & 63) == 0) sh[0][tid >> 6] = b;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < W2; ++w) b = fmaxf(b, (float)sh[0][w]);
      cheb[l] = cheb_of(b);
    }
  }
  __syncthreads();
  turn = 0;

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
      // down
      for (int l = 1; l < L; ++l) {
        const ModalLevelDev &F = M.lev[l - 1], &A = M.lev[l];
        const Vec src = l == 1 ? Z : vec_at(F.t, work), b = vec_at(A.b, work), t = vec_at(A.t, work),
                  y = vec_at(A.y, work);
        const bool last = l == L - 1;
        const Cheb c = cheb[last ? 1 : l];
        for (int i = tid; i < A.n; i += T2) {
          const float v = sell_row(F.R, src, i);
          vset(b, i, v);
          if (!last) vset(t, i, v * c.ith / fmaf(mu, A.area[i], A.diag[i]));
        }
        __syncthreads();
        if (last) break;
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
      // up
      for (int l = L - 2; l >= 1; --l) {
        const ModalLevelDev &A = M.lev[l];
        const Vec yc = vec_at(M.lev[l + 1].y, work), b = vec_at(A.b, work), t = vec_at(A.t, work),
                  y = vec_at(A.y, work);
        const Cheb c = cheb[l];
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
  if (tid == 0) atomicMax(&st->m_cyc, it);
}

int launch_modal_fwd(const Geo &g, hipStream_t s, const ModalDev &M, const double *r, SolverState *st,
                     hipEvent_t *ev) {
  return launch_transform(g, s, M, r, nullptr, st, true, ev);
}

int launch_modal_2d(hipStream_t s, const ModalDev &M, SolverState *st, hipEvent_t *ev) {
  LAUNCH_TIMED(ev, 0, k_modal_2d, dim3(M.nzi), dim3(T2), (size_t)M.lds2d, s, M, st);
  return (int)hipGetLastError();
}

int launch_modal_bwd(const Geo &g, hipStream_t s, const ModalDev &M, double *x, SolverState *st, hipEvent_t *ev) {
  return launch_transform(g, s, M, nullptr, x, st, false, ev);
}

template <int MT>
static bool allow_t(int lds) {
  return hipFuncSetAttribute(reinterpret_cast<const void *>(&k_modal_fwd<MT>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess &&
         hipFuncSetAttribute(reinterpret_cast<const void *>(&k_modal_bwd<MT>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
}

// raises the kernels' dynamic LDS limits to what M asks for
bool modal_allow_lds(const ModalDev &M) {
  const int tr = M.mt * M.kt * 256 * (int)sizeof(double);
  bool ok = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_modal_2d),
                                hipFuncAttributeMaxDynamicSharedMemorySize, M.lds2d) == hipSuccess;
  switch (M.mt) {
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
