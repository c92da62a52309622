// AMReX patch data (FArrayBox) on the device <-> a level's dense node order.
//
// The reference keeps a level's populations, second populations and
// multipliers in MultiFabs (amr_info_holder.f95:50-76): per box an FP64 array
// of ncomp components, component-major, each component the nodal box grown by
// the ghost width, x fastest.  These kernels gather the valid region of such
// an array into [ncomp][n] (node = a + nx (b + ny c)) and scatter it back; the
// ghost cells are neither read nor written.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace uclbs {
namespace {

// element of a FAB component that holds node k of the box
__device__ __forceinline__ int64_t fab_offset(unsigned k, const Box& b, int ghost) {
  const unsigned nx = (unsigned)b.nx, ny = (unsigned)b.ny;
  const unsigned x = k % nx, yz = k / nx, y = yz % ny, z = yz / ny;
  const int64_t gx = b.nx + 2 * ghost, gy = b.ny + 2 * ghost;
  return (int64_t)x + ghost + gx * ((int64_t)y + ghost + gy * ((int64_t)z + ghost));
}

__global__ __launch_bounds__(256) void k_fab_gather(const double* __restrict__ fab, int ghost,
                                                    int64_t cstride, Box b, int ncomp,
                                                    double* __restrict__ dense) {
  const int64_t n = b.n, tot = n * ncomp;
  const int64_t gx = b.nx + 2 * ghost, gy = b.ny + 2 * ghost;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < tot;
       k += (int64_t)gridDim.x * blockDim.x) {
    const int64_t comp = k / n, node = k - comp * n;
    const int64_t a = node % b.nx, yz = node / b.nx, bb = yz % b.ny, c = yz / b.ny;
    dense[k] = fab[comp * cstride + (a + ghost) + gx * ((bb + ghost) + gy * (c + ghost))];
  }
}

// FAB -> level state in storage form, both population buffers in one pass:
// dst0 and dst1[c * n + node] = (S)(fab - ref[c]) (dst1 may be null).  One
// thread takes kGroup components of one node: the node's coordinates are
// formed once and the kGroup loads (8 B a lane, whole wavefront rows) are in
// flight together.  Bound by HBM: 8 + 2 sizeof(S) B per value.  Going through
// a dense FP64 copy (a second pass, a copy into the other buffer, and the
// allocation of that copy on every call) import and export of a 256^3 D3Q27
// level took 7.2 ms together where they take 2.4 ms in this form, and 20
// steps between the two took 21.7 ms a pass, now 16.4 ms, and 204 ms when three
// contexts took turns: their 3.6 GB allocations were returned and mapped anew
// each time.
template <typename S, int kGroup>
__global__ __launch_bounds__(256) void k_fab_import(const double* __restrict__ fab, int ghost,
                                                    int64_t cstride, Box b, FabRef ref,
                                                    S* __restrict__ dst0, S* __restrict__ dst1) {
  const unsigned k = blockIdx.x * 256u + threadIdx.x, n = (unsigned)b.n;
  if (k >= n) return;
  const double* __restrict__ src = fab + fab_offset(k, b, ghost);
  const unsigned c0 = blockIdx.y * kGroup;
  double v[kGroup];
#pragma unroll
  for (int j = 0; j < kGroup; ++j)
    v[j] = __builtin_nontemporal_load(src + (int64_t)(c0 + j) * cstride);
#pragma unroll
  for (int j = 0; j < kGroup; ++j) {
    const S s = (S)(v[j] - ref.v[c0 + j]);
    const size_t at = (size_t)(c0 + j) * n + k;
    dst0[at] = s;
    if (dst1) __builtin_nontemporal_store(s, dst1 + at);
  }
}

// level state -> FAB: fab = src[c * n + node] + ref[c], split as the import
template <typename S, int kGroup>
__global__ __launch_bounds__(256) void k_fab_export(const S* __restrict__ src, int ghost,
                                                    int64_t cstride, Box b, FabRef ref,
                                                    double* __restrict__ fab) {
  const unsigned k = blockIdx.x * 256u + threadIdx.x, n = (unsigned)b.n;
  if (k >= n) return;
  double* __restrict__ dst = fab + fab_offset(k, b, ghost);
  const unsigned c0 = blockIdx.y * kGroup;
  S v[kGroup];
#pragma unroll
  for (int j = 0; j < kGroup; ++j) v[j] = src[(size_t)(c0 + j) * n + k];
#pragma unroll
  for (int j = 0; j < kGroup; ++j)
    __builtin_nontemporal_store((double)v[j] + ref.v[c0 + j], dst + (int64_t)(c0 + j) * cstride);
}

// Plot3D IBLANK of the valid region from the node codes (plot3d_output.f95:
// 275-281): 1 for a fluid node (code >= 0), -1 for code -666, 0 otherwise; 1
// everywhere when the level has no link table (code null)
__global__ __launch_bounds__(256) void k_blank_gather(const int32_t* __restrict__ code, int ghost,
                                                      Box b, int32_t* __restrict__ blank) {
  const int64_t gx = b.nx + 2 * ghost, gy = b.ny + 2 * ghost;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < b.n;
       k += (int64_t)gridDim.x * blockDim.x) {
    int32_t v = 1;
    if (code) {
      const int64_t a = k % b.nx, yz = k / b.nx, bb = yz % b.ny, c = yz / b.ny;
      const int32_t s = code[(a + ghost) + gx * ((bb + ghost) + gy * (c + ghost))];
      v = s >= 0 ? 1 : (s == -666 ? -1 : 0);
    }
    blank[k] = v;
  }
}

__global__ __launch_bounds__(256) void k_fill(double* __restrict__ p, int64_t n, double v) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x)
    p[k] = v;
}

unsigned fab_grid(const Box& b, int ncomp) {
  const int64_t blocks = (b.n * ncomp + 255) / 256;
  return (unsigned)(blocks < 65536 ? blocks : 65536);
}

}  // namespace

hipError_t launch_fab_gather(const double* fab, int ghost, int64_t cstride, const Box& b,
                             int ncomp, double* dense, hipStream_t s) {
  hipLaunchKernelGGL(k_fab_gather, dim3(fab_grid(b, ncomp)), dim3(256), 0, s, fab, ghost, cstride,
                     b, ncomp, dense);
  return hipGetLastError();
}

// components in groups of 9 (27) or 13 (39 and the 13 multipliers): 2-D grid,
// nodes by component groups
hipError_t launch_fab_import(const double* fab, int ghost, int64_t cstride, const Box& b,
                             int ncomp, const FabRef& ref, int fp32, void* dst0, void* dst1,
                             hipStream_t s) {
  const unsigned nb = (unsigned)((b.n + 255) / 256);
  const int group = ncomp == 27 ? 9 : 13;
  if (ncomp % group) return hipErrorInvalidValue;
  const dim3 g(nb, (unsigned)(ncomp / group)), t(256);
#define UCLBS_FAB_IN(S, G)                                                              \
  hipLaunchKernelGGL((k_fab_import<S, G>), g, t, 0, s, fab, ghost, cstride, b, ref,     \
                     static_cast<S*>(dst0), static_cast<S*>(dst1))
  if (fp32) { if (group == 9) UCLBS_FAB_IN(float, 9); else UCLBS_FAB_IN(float, 13); }
  else { if (group == 9) UCLBS_FAB_IN(double, 9); else UCLBS_FAB_IN(double, 13); }
#undef UCLBS_FAB_IN
  return hipGetLastError();
}

hipError_t launch_fab_export(const void* src, const Box& b, int ncomp, const FabRef& ref,
                             int fp32, int ghost, int64_t cstride, double* fab, hipStream_t s) {
  const unsigned nb = (unsigned)((b.n + 255) / 256);
  const int group = ncomp == 27 ? 9 : 13;
  if (ncomp % group) return hipErrorInvalidValue;
  const dim3 g(nb, (unsigned)(ncomp / group)), t(256);
#define UCLBS_FAB_OUT(S, G)                                                             \
  hipLaunchKernelGGL((k_fab_export<S, G>), g, t, 0, s, static_cast<const S*>(src), ghost, \
                     cstride, b, ref, fab)
  if (fp32) { if (group == 9) UCLBS_FAB_OUT(float, 9); else UCLBS_FAB_OUT(float, 13); }
  else { if (group == 9) UCLBS_FAB_OUT(double, 9); else UCLBS_FAB_OUT(double, 13); }
#undef UCLBS_FAB_OUT
  return hipGetLastError();
}

hipError_t launch_blank_gather(const int32_t* code, int ghost, const Box& b, int32_t* blank,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_blank_gather, dim3(fab_grid(b, 1)), dim3(256), 0, s, code, ghost, b, blank);
  return hipGetLastError();
}

hipError_t launch_fill(double* p, int64_t n, double v, hipStream_t s) {
  Box b{};
  b.n = n;
  hipLaunchKernelGGL(k_fill, dim3(fab_grid(b, 1)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

}  // namespace uclbs
