// Entropic over-relaxation parameter alpha: device-side root-finder.
//
// alpha is the nontrivial root of the entropy equality H(f + alpha*D) = H(f),
// D = feq - f, following the Newton definition of the reference
// (looping/timestepping/calculate_alpha.f95:416-556, commented out there):
// positivity bracket alpha_max = min_{D_i<0} -f_i/D_i (:424-445), the rule
// "alpha_max < 2 => alpha = alpha_max" (:449-455) and the clamp to alpha_max
// (:529-536).  Two changes make it safe on a GPU: a bracket with bisection
// fallback and an iteration cap, and the entropy function is evaluated in the
// conditioned form
//     g(a)  = sum_i f_i [(1 + a x_i) ln(1 + a x_i) - a x_i - a x_i ln(1 + x_i)],
//     g'(a) = sum_i D_i [ln(1 + a x_i) - ln(1 + x_i)],     x_i = D_i / f_i,
// which equals H(f + aD) - H(f) when D conserves mass and momentum and
// ln(feq_i / w_i) is affine in c_i (true for the D3Q27 product-form
// equilibrium).  The term -a x_i sums to -a sum(D) = 0 in exact arithmetic;
// keeping it inside phi(y) = (1+y) ln(1+y) - y stops the FP64 rounding of the
// conserved moments of feq from biasing the root.  For max|x_i| small the same g is evaluated from the power
// sums S_n = sum_i f_i x_i^n:
//     g(a)  = sum_{n>=2} (-1)^n S_n (a^n/(n(n-1)) - a/(n-1)),
//     g'(a) = sum_{n>=2} (-1)^n S_n (a^(n-1) - 1)/(n-1),
// truncated at an order whose remainder is below FP64 round-off for the
// node's max|x_i|; each Newton iteration then costs O(order) scalar FP64 work
// instead of 27 logarithms.  All of it runs in FP64.
#pragma once
#include <hip/hip_runtime.h>

#include "far_terms.h"

namespace uclbs {

enum : int { ALPHA_NEWTON = 0, ALPHA_TRIVIAL = 1, ALPHA_BOUND = 2, ALPHA_NONPOS = 3,
             ALPHA_NOCONV = 4, ALPHA_DEFER = 5 /* left to the far-from-equilibrium kernel */ };

struct AlphaOut {
  double alpha;
  int iters;
  int status;
  bool logpath = false;  // g needed direct logarithms (max|x| beyond the series range)
  bool fallback = false; // the learned start failed and the plain start (alpha = 2) ran
};

// below this max|x| the node is at equilibrium and alpha = 2 (the "fi = fieq"
// branch, calculate_alpha.f95:430-431 and :551-556)
constexpr double kTrivialX = 1e-12;

// Largest max|x| for which the order-N truncation of the power-sum series is
// used.  The remainder of g relative to S2 is about (2.2 m)^(N-1) / (N(N-1))
// for Newton iterates a <= 2.2; the host sets the bound from a target eps
// (1e-16 in FP64 mode, i.e. exact to round-off; tol / 2 in FP32 mode, so
// truncation adds at most half the Newton tolerance to the residual of g).
struct SeriesThr {
  double m7, m10, m16;      // FP64 storage: orders 7, 10, 16
  float m_fast;             // order kFastOrder of the fused FP32-storage pass
  float m_mid;              // order kMidOrder, the second in-register tier
};
template <int N>
struct Order {
  static constexpr int value = N;
};
constexpr int kFastOrder = 6;
constexpr int kMidOrder = 12;
inline double series_limit(int N, double eps) {
  return __builtin_pow(eps * N * (N - 1.0), 1.0 / (N - 1.0)) / 2.2;
}
inline SeriesThr make_series_thr(double eps) {
  return SeriesThr{series_limit(7, eps), series_limit(10, eps), series_limit(16, eps), (float)series_limit(kFastOrder, eps),
                   (float)series_limit(kMidOrder, eps)};
}

// 1/v for a normal v: the hardware estimate and two Newton steps (each at
// least doubles the correct bits), within an ulp or so of the quotient
__device__ __forceinline__ double drcp(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = fma(fma(-v, r, 1.0), r, r);
  r = fma(fma(-v, r, 1.0), r, r);
  return r;
}

// 1/v for a value that is rounded to FP32 next: one Newton step on the estimate
// (2^-23 or better), whose 2^-46 that rounding hides
__device__ __forceinline__ double drcp_to_f32(double v) {
  const double r = __builtin_amdgcn_rcp(v);
  return r * (2.0 - v * r);
}

// ln(1 + x) for x > -1 in FP64, about 30 VALU operations: u = 1 + x = 2^e m
// with m in [sqrt(1/2), sqrt(2)), ln m = 2 atanh(s), s = (m-1)/(m+1), |s| <=
// 0.1716, summed to s^23 (remainder < 1e-18); ln 2 split in a high part exact
// in e*ln2_hi and a low part; the rounding error of 1 + x is removed to first
// order, ln(1+x) = ln(u) - ((u - 1) - x)/u.  Reciprocals for both quotients: s
// only needs relative accuracy (its error enters ln as 2 ds), and c/u is a
// correction of size eps.
__device__ __forceinline__ double log1p_dev(double x) {
  const double u = 1.0 + x;
  const double c = (u - 1.0) - x;
  int e;
  double m = __builtin_frexp(u, &e);
  if (m < 0.70710678118654752440) {
    m *= 2.0;
    e -= 1;
  }
  const double s = (m - 1.0) * drcp(m + 1.0);
  const double s2 = s * s;
  double p = 2.0 / 23.0;
  p = p * s2 + 2.0 / 21.0;
  p = p * s2 + 2.0 / 19.0;
  p = p * s2 + 2.0 / 17.0;
  p = p * s2 + 2.0 / 15.0;
  p = p * s2 + 2.0 / 13.0;
  p = p * s2 + 2.0 / 11.0;
  p = p * s2 + 2.0 / 9.0;
  p = p * s2 + 2.0 / 7.0;
  p = p * s2 + 2.0 / 5.0;
  p = p * s2 + 2.0 / 3.0;
  p = p * s2 + 2.0;
  const double ln2_hi = 6.93147180369123816490e-01;  // 0x3FE62E42FEE00000, 32 significant bits
  const double ln2_lo = 1.90821492927058770002e-10;
  const double de = (double)e;
  return de * ln2_hi + (de * ln2_lo + s * p) - c * __builtin_amdgcn_rcp(u);
}

// ln(1 + y) for y > -1 through a 64-entry table over the mantissa: u = 1 + y
// = m 2^e with m in [1, 2), c_k = 1 + (k + 1/2)/64 the centre of m's 1/64
// interval, inv_k = 1/c_k, r = m inv_k - 1 (|r| < 1/128, one FMA) and
// ln u = e ln 2 + L_k + ln(1 + r), L_k = -ln(inv_k), ln(1 + r) by its series
// to r^7 (|r|^8 / 8 < 2e-18).  The rounding of 1 + y is not corrected, so
// the absolute error is up to 1.2e-16: in g = sum f ((1+y) ln(1+y) - y) it
// stays below the acceptance |g| <= tol S2 (tol 1e-10) while S2 > 1e-5 rho,
// as on the far nodes this serves; a node below would report no convergence,
// not a wrong root.  12 FP64 operations, a few on the high word and two
// table reads where log1p_dev takes about 30.
struct LogTable {
  double inv[64], L[64];
};
// entry k of the table (one lane per entry)
__device__ __forceinline__ void log_table_entry(LogTable& t, int k) {
  const double inv = 1.0 / (1.0 + (k + 0.5) / 64.0);
  t.inv[k] = inv;
  t.L[k] = -log1p_dev(inv - 1.0);  // inv in (0.5, 1): inv - 1 is exact
}
__device__ __forceinline__ double log1p_tab(double y, const LogTable& t) {
  const double u = 1.0 + y;
  // exponent, top six bits of the mantissa and m from the high word (u normal)
  const int hi = __double2hiint(u);
  const int k = (hi >> 14) & 63;
  const double m = __hiloint2double((hi & 0x000fffff) | 0x3ff00000, __double2loint(u));
  const double r = fma(m, t.inv[k], -1.0);
  double p = 1.0 / 7.0;
  p = fma(p, r, -1.0 / 6.0);
  p = fma(p, r, 1.0 / 5.0);
  p = fma(p, r, -0.25);
  p = fma(p, r, 1.0 / 3.0);
  p = fma(p, r, -0.5);
  p = fma(p, r, 1.0);
  const double ln2_hi = 6.93147180369123816490e-01;
  const double ln2_lo = 1.90821492927058770002e-10;
  const double de = (double)((hi >> 20) - 1023);
  return fma(de, ln2_hi, t.L[k]) + fma(p, r, de * ln2_lo);
}

// The series as a polynomial: with C_n = (-1)^n S_n / (n (n-1)) and
// L = sum (-1)^n S_n / (n-1),
//     g(a) = a^2 Q(a) - L a,  g'(a) = a (2 Q(a) + a Q'(a)) - L,  Q = sum C_n a^(n-2),
// so that an evaluation is two FMAs an order (Horner and its derivative) and
// the coefficient's product where the terms one by one take six operations an
// order.  sn(n) yields S_n; the coefficients are formed as they are used, since
// keeping them (2 N registers) would cost the FP32 kernels their occupancy.
template <int N, class SN>
struct SeriesPoly {
  SN sn;
  double L;
  __device__ __forceinline__ explicit SeriesPoly(SN s) : sn(s), L(0.0) {
#pragma unroll
    for (int n = N; n >= 2; --n) L = fma(sn(n), ((n & 1) ? -1.0 : 1.0) / (n - 1.0), L);
  }
  __device__ __forceinline__ void operator()(double a, double& g, double& gp) const {
    double q = sn(N) * (((N & 1) ? -1.0 : 1.0) / (N * (N - 1.0))), dq = 0.0;
#pragma unroll
    for (int n = N - 1; n >= 2; --n) {
      dq = fma(dq, a, q);
      q = fma(q, a, sn(n) * (((n & 1) ? -1.0 : 1.0) / (n * (n - 1.0))));
    }
    const double aq = a * q;
    g = a * (aq - L);
    gp = fma(a, fma(a, dq, q + q), -L);
  }
};
template <int N, class SN>
__device__ __forceinline__ SeriesPoly<N, SN> series_poly(SN sn) {
  return SeriesPoly<N, SN>(sn);
}

// Safeguarded Newton shared by both evaluations of g.  Iterations count Newton
// updates taken before |g(a)| <= tol * S2 (S2 = sum f x^2 ~ g'(root), so the
// test bounds |a - root| by about tol).
template <class Eval>
__device__ __forceinline__ AlphaOut newton_alpha(Eval&& ev, double S2, double amax,
                                                 double alpha0, double tol, int maxit) {
  double lo = 1.0, hi = amax < 1e6 ? amax : 1e6;
  bool hi_is_bound = amax < 1e6;
  double a = (alpha0 > lo && alpha0 < hi) ? alpha0 : 2.0;
  AlphaOut r{2.0, 0, ALPHA_NEWTON, false};
  for (int k = 0;; ++k) {
    double g, gp;
    ev(a, g, gp);
    if (fabs(g) <= tol * S2) { r.alpha = a; r.iters = k; return r; }
    if (g < 0.0 && a >= amax) { r.alpha = amax; r.iters = k; r.status = ALPHA_BOUND; return r; }
    if (k >= maxit) { r.alpha = a; r.iters = k; r.status = ALPHA_NOCONV; return r; }
    if (g < 0.0) lo = a; else { hi = a; hi_is_bound = false; }
    // (a zero or infinite g' gives NaN: the middle of the bracket)
    double an = fma(-g, drcp(gp), a);
    if (!(an > lo && an < hi)) an = (hi_is_bound && an >= hi) ? amax : 0.5 * (lo + hi);
    if (an == amax) hi_is_bound = false;
    a = an;
  }
}

// Root of g for a node far from equilibrium, from sweeps of logarithms at a
// centre a0 and the exact re-expansion of g about it.  With d = a - a0,
// A_i = 1 + a0 x_i and z_i = x_i / A_i, 1 + a x_i = A_i (1 + d z_i) and
//   g(a0 + d) = g(a0) + g'(a0) d + sum_{n>=2} (-1)^n T_n d^n / (n(n-1)),
//   T_n = sum_i D_i z_i^(n-1),
// from (1+t) ln(1+t) = t + sum_{n>=2} (-1)^n t^n / (n(n-1)) at t = d z_i and
// f_i A_i z_i^n = D_i z_i^(n-1).  Since D_i z_i = f_i x_i^2 / A_i >= 0,
// |T_n| <= zmax^(n-2) T_2 and the orders beyond N add at most
//   R = T_2 d^2 (|d| zmax)^(N-1) / (N (N+1) (1 - |d| zmax)).
// One sweep (Q logarithms) gives g(a0), g'(a0) and T_2..T_N; Newton on the
// order-N polynomial (scalar work) gives d, and a0 + d is the root when the
// polynomial's residual plus R plus what the FP32 rounding of the T_n can add
// (far_terms.h) is within tol * S2.  Otherwise the next sweep
// is centred at a0 + d, kept inside the Newton bracket and within
// |d| zmax <= 1/2.  From a seed near the root one sweep suffices where Newton
// on direct logarithms evaluates g two to four times.  Bracket, bound and
// iteration cap follow newton_alpha; iters counts the updates of the centre
// or of the accepted root, as Newton counts its updates.
// sweep(a, w, first) fills a Sweep; the first one also gives K = sum D ln(1 + x)
// (every lane's first sweep is the same one, so that the branch is uniform).
template <int N>
struct Sweep : FarTerms<N> {
  double K;
  double g, gp;  // sum f ((1 + y) ln(1 + y) - y) and sum D ln(1 + y), y = a x
  bool edge;     // a at the positivity bound: some 1 + a x_i <= 0
};
template <int N, class SW>
__device__ __forceinline__ AlphaOut recentred_alpha(SW&& sweep, double S2, double amax,
                                                    double alpha0, double tol, int maxit) {
  double lo = 1.0, hi = amax < 1e6 ? amax : 1e6;
  bool hi_is_bound = amax < 1e6;
  double a = (alpha0 > lo && alpha0 < hi) ? alpha0 : 2.0;
  AlphaOut r{2.0, 0, ALPHA_NEWTON, true};
  Sweep<N> w;
  for (int k = 0;; ++k) {
    sweep(a, w, k == 0);
    const double g = fma(-a, w.K, w.g), gp = w.gp - w.K;
    const double zmax = w.zbound();
    if (fabs(g) <= tol * S2) { r.alpha = a; r.iters = k; return r; }
    if (g < 0.0 && a >= amax) { r.alpha = amax; r.iters = k; r.status = ALPHA_BOUND; return r; }
    if (k >= maxit) { r.alpha = a; r.iters = k; r.status = ALPHA_NOCONV; return r; }
    if (g < 0.0) lo = a; else { hi = a; hi_is_bound = false; }
    if (w.edge) { a = 0.5 * (lo + hi); continue; }
    // Newton on the polynomial p(d) = g + gp d + d^2 Q(d), Q = sum C_n d^(n-2),
    // C_n = (-1)^n T_n / (n (n-1)), from d = 0, |d| within the trust radius
    const double rad = zmax > 0.0 ? 0.5 * drcp(zmax) : 1e300;
    double dl = lo - a, dh = hi - a;
    double dd = 0.0, p = g, pd = gp;
    bool ok = true;
    for (int j = 0; j < 8; ++j) {
      const double st = fma(-p, drcp(pd), dd);
      if (!(st > dl && st < dh) || fabs(st) > rad) { ok = false; dd = st; break; }
      dd = st;
      double q = (double)w.T[N] * (((N & 1) ? -1.0 : 1.0) / (N * (N - 1.0))), dq = 0.0;
#pragma unroll
      for (int n = N - 1; n >= 2; --n) {
        dq = fma(dq, dd, q);
        q = fma(q, dd, (double)w.T[n] * (((n & 1) ? -1.0 : 1.0) / (n * (n - 1.0))));
      }
      const double dQ = dd * q;
      p = fma(dd, dQ + gp, g);
      pd = fma(dd, fma(dd, dq, q + q), gp);
      if (fabs(p) <= 0.25 * tol * S2) break;
    }
    const double q = fabs(dd) * zmax;
    double rem = 1e300;
    if (ok && q < 0.5) {
      double qp = 1.0;
#pragma unroll
      for (int n = 0; n < N - 1; ++n) qp *= q;
      rem = (double)w.T[2] * dd * dd * qp * (1.0 / (N * (N + 1.0))) * drcp(1.0 - q);
      rem += w.slack(dd);
    }
    if (ok && fabs(p) + rem <= tol * S2) { r.alpha = a + dd; r.iters = k + 1; return r; }
    // next centre: the polynomial's step where it stays in the bracket and the
    // trust radius, else the bound or the middle of the bracket
    double an = a + (fabs(dd) > rad ? (dd > 0.0 ? rad : -rad) : dd);
    if (!(an > lo && an < hi)) an = (hi_is_bound && an >= hi) ? amax : 0.5 * (lo + hi);
    if (an == amax) hi_is_bound = false;
    a = an;
  }
}

// S_2..S_N of f x^n = D x^(n-1) over the 27 directions: two orders share a
// product, D x^(2k) times x and times x^2
template <int N>
__device__ __forceinline__ void power_sums27(const double (&D)[27], const double (&x)[27],
                                             double (&S)[N + 1]) {
#pragma unroll
  for (int n = 2; n <= N; ++n) S[n] = 0.0;
#pragma unroll
  for (int i = 0; i < 27; ++i) {
    const double y = x[i] * x[i];
    double t = D[i];
#pragma unroll
    for (int n = 2; n <= N; n += 2) {
      S[n] = fma(t, x[i], S[n]);
      if (n < N) S[n + 1] = fma(t, y, S[n + 1]);
      if (n + 2 <= N) t *= y;
    }
  }
}

// alpha of an FP64 node from D_i, x_i = D_i / f_i, m = max|x|, xmin = min x.
// The lanes of a wavefront run one Newton on series of the largest order that
// one of them needs; a lane that needs fewer terms has zeros for the others, so
// that its alpha is its own order's to the bit, whatever its neighbours need.  A
// lane beyond order 16 takes direct logarithms.
__device__ __forceinline__ AlphaOut solve_alpha27(const double (&f)[27], const double (&D)[27],
                                                  const double (&x)[27], bool nonpos, double m,
                                                  double xmin, double alpha0, double tol, int maxit,
                                                  const SeriesThr& thr) {
  const double amax = xmin < 0.0 ? -1.0 / xmin : 1e300;
  AlphaOut r{2.0, 0, ALPHA_TRIVIAL, false};
  bool open = false;
  if (nonpos) r.status = ALPHA_NONPOS;
  else if (m < kTrivialX) r.status = ALPHA_TRIVIAL;
  else if (amax < 2.0) r = AlphaOut{amax, 0, ALPHA_BOUND, false};
  else open = true;
  auto series = [&](auto order) __attribute__((always_inline)) {
    constexpr int N = decltype(order)::value;
    double S[N + 1];
    power_sums27<N>(D, x, S);
    // products, not selects: around selects the compiler spills 300 registers
    const double keep10 = m > thr.m7 ? 1.0 : 0.0, keep16 = m > thr.m10 ? 1.0 : 0.0;
#pragma unroll
    for (int n = 8; n <= N; ++n) S[n] *= n > 10 ? keep16 : keep10;
    const auto ev = series_poly<N>([&](int n) __attribute__((always_inline)) { return S[n]; });
    if (open && m <= thr.m16) r = newton_alpha(ev, S[2], amax, alpha0, tol, maxit);
  };
  const bool wide = open && m > thr.m7 && m <= thr.m16;
  if (__any(wide && m > thr.m10)) series(Order<16>());
  else if (__any(wide)) series(Order<10>());
  else if (__any(open && m <= thr.m16)) series(Order<7>());
  if (open && !(m <= thr.m16)) {
    // g(a) = sum f ((1 + y) ln(1 + y) - y) - a K, y = a x, K = sum D ln(1 + x);
    // (1+y) ln(1+y) - y loses only absolute accuracy O(eps |y|), far below
    // tol * S2
    double K = 0.0, S2 = 0.0;
#pragma unroll
    for (int i = 0; i < 27; ++i) {
      K = fma(D[i], log1p_dev(x[i]), K);
      S2 = fma(D[i], x[i], S2);
    }
    r = newton_alpha(
        [&](double a, double& g, double& gp) __attribute__((always_inline)) {
          double sg = 0.0, sgp = 0.0;
          bool inf_gp = false;
#pragma unroll
          for (int i = 0; i < 27; ++i) {
            const double y = a * x[i], u = 1.0 + y;
            if (u <= 0.0) { sg -= f[i] * y; inf_gp = true; continue; }  // limit of u ln u at 0
            const double la = log1p_dev(y);
            sg = fma(f[i], fma(u, la, -y), sg);
            sgp = fma(D[i], la, sgp);
          }
          g = fma(-a, K, sg);
          gp = inf_gp ? __builtin_huge_val() : sgp - K;
        },
        S2, amax, alpha0, tol, maxit);
    r.logpath = true;
  }
  return r;
}

}  // namespace uclbs
