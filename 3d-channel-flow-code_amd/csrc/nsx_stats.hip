// nsx_stats.hip -- channel turbulence statistics of the reference
// (src/Stats/stats.F90) on the resident fields: the twelve running sums of
// glob_sample and the plane sums of glob_put_plane_mm (in its summation
// order); nsx_files.hip writes the files.
//
// Layout: the accumulators are cell fields, double[N0][NS] like every other
// cell field of the library, and cover the layers k = 0..NZ-1 (ghost layers
// included, as glob_sample's loop does).
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "nsx_kernels.h"

// glob_sample, stats.F90:142-174: every column i < N_CELL0 and every layer
// (k = 1..NZ of the reference), in its operation order
__global__ __launch_bounds__(NSX_BLOCK) void k_glob_sample(Geo g, const double *u, const double *v,
                                                            const double *w, const double *p, const double *eddy,
                                                            StatsBufs sm) {
  const size_t n = (size_t)g.N0 * g.NS;
  for (size_t t = (size_t)blockIdx.x * NSX_BLOCK + threadIdx.x; t < n; t += (size_t)gridDim.x * NSX_BLOCK) {
    const int k = (int)(t % (size_t)g.NS);
    if (k >= g.NZ) continue;
    const double tu = u[t], tv = v[t], tw = w[t], tp = p[t];
    const double tp2 = tp * tp, tu2 = tu * tu, tv2 = tv * tv, tw2 = tw * tw;
    const double tuv = tu * tv, tvw = tv * tw, twu = tw * tu;
    sm.a[SM_UF][t] = sm.a[SM_UF][t] + tu;
    sm.a[SM_VF][t] = sm.a[SM_VF][t] + tv;
    sm.a[SM_WF][t] = sm.a[SM_WF][t] + tw;
    sm.a[SM_PF][t] = sm.a[SM_PF][t] + tp;
    sm.a[SM_U2F][t] = sm.a[SM_U2F][t] + tu2;
    sm.a[SM_V2F][t] = sm.a[SM_V2F][t] + tv2;
    sm.a[SM_W2F][t] = sm.a[SM_W2F][t] + tw2;
    sm.a[SM_UVF][t] = sm.a[SM_UVF][t] + tuv;
    sm.a[SM_VWF][t] = sm.a[SM_VWF][t] + tvw;
    sm.a[SM_WUF][t] = sm.a[SM_WUF][t] + twu;
    sm.a[SM_P2F][t] = sm.a[SM_P2F][t] + tp2;
    if (eddy) sm.a[SM_EF][t] = sm.a[SM_EF][t] + eddy[t];
  }
}

// glob_put_plane_mm, stats.F90:266-279: S_q(k) = sum over i = 1..N_CELL0, in
// order, of sm_q(i,k)/ns, for the nine velocity moments and the interior
// layers.  Each sum is a serial chain of N_CELL0 additions in the
// reference's sequence, so the kernel is bound by that chain and by how the
// columns reach it: a block takes PL layers (a column's are one 32-byte run,
// instead of 8 bytes of every column); wave 0, a lane per sum, adds a
// tile of PC columns while the other waves write the next one, divided by ns,
// and have the one after in flight.  65,536 columns x 96 layers: 3.57 ms with a
// layer a block, its divisions in the chain and no overlap, now 1.5; 16,384 x
// 64: 0.88 and 0.30.
constexpr int PL = 4, PC = 256, PSTR = PC + 2, PT = 1024;
constexpr int PITEMS = (SM_NPLANE * PC + PT - 65) / (PT - 64);
constexpr size_t PLANE_LDS = 2 * sizeof(double) * SM_NPLANE * PL * PSTR;

__global__ __launch_bounds__(PT) void k_plane_sums(Geo g, StatsBufs sm, double ns, double *out) {
  extern __shared__ __align__(16) unsigned char nsx_dyn_lds[];
  double(*tile)[PSTR] = reinterpret_cast<double(*)[PSTR]>(nsx_dyn_lds);  // two of SM_NPLANE * PL rows
  // an XCD's blocks take adjacent layers: their runs share cache lines
  const int G = gridDim.x, b = blockIdx.x;
  const int lb = G % NSX_NXCD == 0 ? (b % NSX_NXCD) * (G / NSX_NXCD) + b / NSX_NXCD : b;
  const int k0 = 1 + PL * lb, nl = min(PL, g.NZ - 1 - k0);
  const int q = threadIdx.x, ntile = (g.N0 + PC - 1) / PC;
  const bool adds = q < SM_NPLANE * PL && q % PL < nl;
  double v[PITEMS][PL];
  auto fetch = [&](int t) {
#pragma unroll
    for (int n = 0; n < PITEMS; ++n) {
      const int w = q - 64 + n * (PT - 64), r = w / PC, i = t * PC + w % PC;
#pragma unroll
      for (int l = 0; l < PL; ++l) v[n][l] = 0.0;
      if (r >= SM_NPLANE || i >= g.N0) continue;
      // two 16-byte loads: a wave's loads touch a line per lane each, and
      // their number bounds the fetch (8-byte ones: 3.06 ms)
      const double *src = sm.a[r] + (size_t)i * g.NS + k0;
      if (nl == PL)
        __builtin_memcpy(v[n], src, PL * sizeof(double));
      else
#pragma unroll
        for (int l = 0; l < PL; ++l)
          if (l < nl) v[n][l] = src[l];
    }
  };
  auto store = [&](int t) {
#pragma unroll
    for (int n = 0; n < PITEMS; ++n) {
      const int w = q - 64 + n * (PT - 64), r = w / PC;
      if (r < SM_NPLANE)
#pragma unroll
        for (int l = 0; l < PL; ++l) tile[(t & 1) * SM_NPLANE * PL + r * PL + l][w % PC] = v[n][l] / ns;
    }
  };
  if (q >= 64) {
    fetch(0);
    store(0);
    fetch(1);
  }
  __syncthreads();
  double s = 0.0;
  for (int t = 0; t < ntile; ++t) {
    if (q >= 64) {
      store(t + 1);
      fetch(t + 2);
    } else if (adds) {
      const double *a = tile[(t & 1) * SM_NPLANE * PL + q];
      const int m = min(PC, g.N0 - t * PC);
      int j = 0;
      for (; j + 16 <= m; j += 16) {
        double b[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) b[u] = a[j + u];
#pragma unroll
        for (int u = 0; u < 16; ++u) s = s + b[u];
      }
      for (; j < m; ++j) s = s + a[j];
    }
    __syncthreads();
  }
  if (adds) out[(size_t)(q / PL) * g.NZ + k0 + q % PL] = s;
}

int launch_glob_sample(const Geo &g, hipStream_t s, const double *u, const double *v, const double *w,
                       const double *p, const double *eddy, StatsBufs sm) {
  const size_t n = (size_t)g.N0 * g.NS;
  size_t blocks = (n + NSX_BLOCK - 1) / NSX_BLOCK;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_glob_sample, dim3((unsigned)blocks), dim3(NSX_BLOCK), 0, s, g, u, v, w, p, eddy, sm);
  return (int)hipGetLastError();
}

int launch_plane_sums(const Geo &g, hipStream_t s, StatsBufs sm, int ns, double *out) {
  if (g.NZ < 3) return 0;
  // two tiles pass the 64 KB that a kernel may have unasked
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_plane_sums),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)PLANE_LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(k_plane_sums, dim3((unsigned)((g.NZ - 2 + PL - 1) / PL)), dim3(PT), PLANE_LDS, s, g, sm, (double)ns,
                     out);
  return (int)hipGetLastError();
}
