// nsx_xfer.hip -- a field's layers between the device layout (column by
// column, layers contiguous) and the reference's (layer by layer, columns
// contiguous) for nsx_put_field and nsx_get_field.
//
// A chunk of layers is transposed through LDS on the device and crosses as
// contiguous rows; bound by the host's copy between its array and the pinned
// chunk.  Transposed on the host (a read or write of 8 bytes every 800 per
// element), a 52 MB field took 21 ms out and 17.5 ms in; now 3.5 and 1.4.
#include "nsx_kernels.h"

constexpr int XT = 32;  // the tile: 32 columns x 32 layers

// out[(k - k0) * w + r] = f[src(r) * stride + k] for the layers k0 .. k0+nk-1
// and the rows r < w; src(r) = r for r < n, else ghost[r - n]
__global__ __launch_bounds__(256) void k_field_out(const double *f, int stride, int k0, int nk, int w, int n,
                                                   const int *ghost, double *out) {
  __shared__ double t[XT][XT + 1];
  const int r0 = blockIdx.x * XT, kb = blockIdx.y * XT;
  for (int q = threadIdx.x; q < XT * XT; q += 256) {
    const int r = r0 + q / XT, k = kb + q % XT;
    if (r < w && k < nk) {
      const int c = r < n ? r : ghost[r - n];
      t[q / XT][q % XT] = f[(size_t)c * stride + k0 + k];
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < XT * XT; q += 256) {
    const int r = r0 + q % XT, k = kb + q / XT;
    if (r < w && k < nk) out[(size_t)k * w + r] = t[q % XT][q / XT];
  }
}

// f[c * stride + k] = in[(k - k0) * w + c] for the layers k0 .. k0+nk-1 of the
// columns c < w; layers at and past kz are zero
__global__ __launch_bounds__(256) void k_field_in(const double *in, int w, int k0, int nk, int kz, int stride,
                                                  double *f) {
  __shared__ double t[XT][XT + 1];
  const int c0 = blockIdx.x * XT, kb = blockIdx.y * XT;
  for (int q = threadIdx.x; q < XT * XT; q += 256) {
    const int c = c0 + q % XT, k = kb + q / XT;
    if (c < w && k < nk) t[q % XT][q / XT] = k0 + k < kz ? in[(size_t)k * w + c] : 0.0;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < XT * XT; q += 256) {
    const int c = c0 + q / XT, k = kb + q % XT;
    if (c < w && k < nk) f[(size_t)c * stride + k0 + k] = t[q / XT][q % XT];
  }
}

int launch_field_out(hipStream_t s, const double *f, int stride, int k0, int nk, int w, int n, const int *ghost,
                     double *out) {
  hipLaunchKernelGGL(k_field_out, dim3((w + XT - 1) / XT, (nk + XT - 1) / XT), dim3(256), 0, s, f, stride, k0, nk, w,
                     n, ghost, out);
  return (int)hipGetLastError();
}

int launch_field_in(hipStream_t s, const double *in, int w, int k0, int nk, int kz, int stride, double *f) {
  hipLaunchKernelGGL(k_field_in, dim3((w + XT - 1) / XT, (nk + XT - 1) / XT), dim3(256), 0, s, in, w, k0, nk, kz,
                     stride, f);
  return (int)hipGetLastError();
}
