// staging.hip -- state arrays to and from pinned host memory in a host layout.
//
// A copy of a state array crosses PCIe once, in FP64 and already in the
// caller's layout: the kernels read (write) the device planes and write (read)
// a pinned staging buffer directly, converting (hi, lo) pairs and floats on
// the way, so the host is left with one contiguous memory copy.  The state is
// cut into chunks of `units`: rows (v, j) of ni values for the plane layouts,
// columns i of nj cells for the [i][j][var] layout, whose transposition goes
// through LDS so that both sides move whole 64-byte lines.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace e2d {

namespace {

// element of a plane <-> FP64 value
__device__ __forceinline__ double get(const double *p, long long k) { return p[k]; }
__device__ __forceinline__ double get(const float2 *p, long long k) {
  const float2 x = p[k];
  return (double)x.x + (double)x.y;
}
__device__ __forceinline__ double get(const float *p, long long k) { return (double)p[k]; }
__device__ __forceinline__ void put(double *p, long long k, double x) { p[k] = x; }
__device__ __forceinline__ void put(float2 *p, long long k, double x) {
  const float hi = (float)x;
  p[k] = make_float2(hi, (float)(x - (double)hi));
}
__device__ __forceinline__ void put(float *p, long long k, double x) { p[k] = (float)x; }

constexpr int kThreads = 256;

// rows [first, first + rows) of the box's 4 x nj rows, ni values each
template <class E, bool TO_HOST>
__global__ __launch_bounds__(kThreads) void rows_kernel(Grid g, HostBox b, int first,
                                                        long long count, double *host) {
  E *p = static_cast<E *>(g.p);
  for (long long k = blockIdx.x * (long long)kThreads + threadIdx.x; k < count;
       k += (long long)gridDim.x * kThreads) {
    const long long row = k / b.ni;
    const int i = (int)(k - row * b.ni);
    const int vj = first + (int)row;
    const int v = vj / b.nj, j = vj - v * b.nj;
    const long long o = v * g.plane + (long long)(b.j0 + j) * g.pitch + b.i0 + i;
    if constexpr (TO_HOST)
      host[k] = get(p, o);
    else
      put(p, o, host[k]);
  }
}

// columns [first, first + cols) of the box as [i][j][var].  A block moves tiles
// of 16 columns x 32 rows x 4 variables: 128-byte row pieces on the device
// side, 1 KiB runs on the host side.
constexpr int kTi = 16, kTj = 32;

template <class E, bool TO_HOST>
__global__ __launch_bounds__(kThreads) void columns_kernel(Grid g, HostBox b, int first, int cols,
                                                           double *host) {
  __shared__ double tile[kTi][kTj * 4 + 2];
  E *p = static_cast<E *>(g.p);
  const int ta = blockIdx.x * kTi, tj = blockIdx.y * kTj;
  const int ni = min(kTi, cols - ta), nj = min(kTj, b.nj - tj);
  auto device_side = [&](auto &&move) {
    for (int k = threadIdx.x; k < kTi * kTj * 4; k += kThreads) {
      const int i = k % kTi, j = (k / kTi) % kTj, v = k / (kTi * kTj);
      if (i < ni && j < nj)
        move(v * g.plane + (long long)(b.j0 + tj + j) * g.pitch + b.i0 + first + ta + i,
             tile[i][j * 4 + v]);
    }
  };
  auto host_side = [&](auto &&move) {
    for (int k = threadIdx.x; k < kTi * kTj * 4; k += kThreads) {
      const int i = k / (kTj * 4), jv = k % (kTj * 4);
      if (i < ni && jv < nj * 4)
        move(((long long)(ta + i) * b.nj + tj) * 4 + jv, tile[i][jv]);
    }
  };
  if constexpr (TO_HOST) {
    device_side([&](long long o, double &t) { t = get(p, o); });
    __syncthreads();
    host_side([&](long long o, double &t) { host[o] = t; });
  } else {
    host_side([&](long long o, double &t) { t = host[o]; });
    __syncthreads();
    device_side([&](long long o, double &t) { put(p, o, t); });
  }
}

template <class E, bool TO_HOST>
void launch_t(Grid g, const HostBox &b, bool columns, int first, int units, double *host,
              hipStream_t st) {
  if (columns) {
    const dim3 grid((units + kTi - 1) / kTi, (b.nj + kTj - 1) / kTj);
    hipLaunchKernelGGL((columns_kernel<E, TO_HOST>), grid, dim3(kThreads), 0, st, g, b, first,
                       units, host);
  } else {
    const long long count = (long long)units * b.ni;
    const long long blocks = (count + kThreads - 1) / kThreads;
    hipLaunchKernelGGL((rows_kernel<E, TO_HOST>), dim3((unsigned)(blocks < 4096 ? blocks : 4096)),
                       dim3(kThreads), 0, st, g, b, first, count, host);
  }
}

}  // namespace

hipError_t launch_staging(int precision, Grid g, const HostBox &b, bool columns, int first,
                          int units, double *host, bool to_host, hipStream_t st) {
  if (units < 1 || first < 0 || first + units > (columns ? b.ni : 4 * b.nj))
    return hipErrorInvalidValue;
#define E2D_STAGE(E)                                                       \
  to_host ? launch_t<E, true>(g, b, columns, first, units, host, st)       \
          : launch_t<E, false>(g, b, columns, first, units, host, st)
  if (precision == E2D_PRECISION_FP32_SPLIT)
    E2D_STAGE(float2);
  else if (precision == E2D_PRECISION_FP32)
    E2D_STAGE(float);
  else
    E2D_STAGE(double);
#undef E2D_STAGE
  return hipGetLastError();
}

}  // namespace e2d
