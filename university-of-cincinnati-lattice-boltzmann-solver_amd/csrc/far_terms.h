// Coefficients of the polynomial that steps a far-from-equilibrium node's
// root-find (alpha_solve.h, recentred_alpha), and what their rounding can do.
// No dependence on HIP beyond the function attributes.
#pragma once

namespace uclbs {

// T_n = sum_i D_i z_i^(n-1), n = 2..N, z_i = x_i / A_i with A_i = 1 + a x_i: the
// polynomial sum (-1)^n T_n d^n / (n (n-1)).  FP32, as they only steer the step
// (g and g' are FP64 and decide acceptance) and as N + 1 FP64 sums would cost
// the kernel its occupancy; z is formed in FP64 and rounded once.
template <int N>
struct FarTerms {
  float T[N + 1];
  float zmax;  // max |z|

  __host__ __device__ __forceinline__ void clear() {
    zmax = 0.0f;
#pragma unroll
    for (int n = 2; n <= N; ++n) T[n] = 0.0f;
  }
  // one direction; rA = 1 / A (0 where A <= 0: it adds nothing)
  __host__ __device__ __forceinline__ void add(float D, double x, double rA) {
    const float z = (float)(x * rA), az = __builtin_fabsf(z);
    zmax = az > zmax ? az : zmax;
    float t = D;
#pragma unroll
    for (int n = 2; n <= N; ++n) {
      t *= z;
      T[n] += t;
    }
  }
  // not below the unrounded max |z|
  __host__ __device__ __forceinline__ double zbound() const { return (double)zmax * (1.0 + 1e-6); }

  // Bound of the polynomial's error at d from the rounding of T.  With u = 2^-24
  // a term of T_n has n - 1 roundings of z and n - 1 of products, the sum of 27
  // terms 26 more, so that T_n is off by at most (26 + 2 (n - 1)) u W_n <= 36 u
  // W_n = 2.15e-6 W_n for n <= 6, W_n = sum |D z^(n-1)|.  D and z have the same
  // sign: W_n = T_n for even n, and W_n <= max|z| W_(n-1) for odd n, where T_n
  // itself may cancel.
  __host__ __device__ __forceinline__ double slack(double d) const {
    static_assert(N <= 6, "rounding count");
    const double a = __builtin_fabs(d), zm = zbound();
    double s = 0.0;
#pragma unroll
    for (int n = N; n >= 2; --n)
      s = __builtin_fma(s, a, (n & 1 ? zm * (double)T[n - 1] : (double)T[n]) * (1.0 / (n * (n - 1.0))));
    return 2.2e-6 * a * a * s;
  }
};

}  // namespace uclbs
