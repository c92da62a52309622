// D3Q39 step of a level without boundaries: every node of a periodic box pulls
// its populations from the box and takes the node update of k_d3q39.hip, with
// the sums over the 39 velocities formed by groups of sign images
// (d3q39_groups.h), exponentials through a table and reciprocals for quotients.
//
// The step is bound by the issue of FP64 instructions at one wavefront a SIMD
// (its 13 x 13 factorisation takes over 300 VGPRs) and by fetching the straight
// code, so what counts is the number of operations: ~1,700 a Newton iteration
// where a product per direction and monomial takes 3,400, ~1,500 for the
// collision where it took 4,500.
//
// 65 x 48 x 33, FP32 storage: 116 -> 83 us a step; 96 x 80 x 64 shifted, FP64
// storage: 861 -> 350 us (there g is not staged in LDS, so that four blocks fit
// a CU instead of two, and is read again ahead of alpha: 399 us where the
// collision waited for it).  Distance from 64-bit results: 1.6e-9 as before, 1.4e-14
// -> 1.2e-14.
//
// Levels with faces, walls or ghost nodes keep k_d3q39.hip's summation order:
// one step differs by 1e-13, but there the repair of negative populations and
// the wall rule jump with the sign of a value near zero, and the difference
// grows (34 steps of the 384 x 192 x 96 wedge: 3e-5), so that a run would not
// repeat its recorded results.
#include "d3q39_groups.h"
#include "d3q39_wave.h"
#include "kernels.h"

#include <type_traits>

namespace uclbs {

namespace {

// 2^(j / 64) to the nearest double
__constant__ const double kExp2_64[64] = {
    0x1.0000000000000p+0, 0x1.02c9a3e778061p+0, 0x1.059b0d3158574p+0, 0x1.0874518759bc8p+0,
    0x1.0b5586cf9890fp+0, 0x1.0e3ec32d3d1a2p+0, 0x1.11301d0125b51p+0, 0x1.1429aaea92de0p+0,
    0x1.172b83c7d517bp+0, 0x1.1a35beb6fcb75p+0, 0x1.1d4873168b9aap+0, 0x1.2063b88628cd6p+0,
    0x1.2387a6e756238p+0, 0x1.26b4565e27cddp+0, 0x1.29e9df51fdee1p+0, 0x1.2d285a6e4030bp+0,
    0x1.306fe0a31b715p+0, 0x1.33c08b26416ffp+0, 0x1.371a7373aa9cbp+0, 0x1.3a7db34e59ff7p+0,
    0x1.3dea64c123422p+0, 0x1.4160a21f72e2ap+0, 0x1.44e086061892dp+0, 0x1.486a2b5c13cd0p+0,
    0x1.4bfdad5362a27p+0, 0x1.4f9b2769d2ca7p+0, 0x1.5342b569d4f82p+0, 0x1.56f4736b527dap+0,
    0x1.5ab07dd485429p+0, 0x1.5e76f15ad2148p+0, 0x1.6247eb03a5585p+0, 0x1.6623882552225p+0,
    0x1.6a09e667f3bcdp+0, 0x1.6dfb23c651a2fp+0, 0x1.71f75e8ec5f74p+0, 0x1.75feb564267c9p+0,
    0x1.7a11473eb0187p+0, 0x1.7e2f336cf4e62p+0, 0x1.82589994cce13p+0, 0x1.868d99b4492edp+0,
    0x1.8ace5422aa0dbp+0, 0x1.8f1ae99157736p+0, 0x1.93737b0cdc5e5p+0, 0x1.97d829fde4e50p+0,
    0x1.9c49182a3f090p+0, 0x1.a0c667b5de565p+0, 0x1.a5503b23e255dp+0, 0x1.a9e6b5579fdbfp+0,
    0x1.ae89f995ad3adp+0, 0x1.b33a2b84f15fbp+0, 0x1.b7f76f2fb5e47p+0, 0x1.bcc1e904bc1d2p+0,
    0x1.c199bdd85529cp+0, 0x1.c67f12e57d14bp+0, 0x1.cb720dcef9069p+0, 0x1.d072d4a07897cp+0,
    0x1.d5818dcfba487p+0, 0x1.da9e603db3285p+0, 0x1.dfc97337b9b5fp+0, 0x1.e502ee78b3ff6p+0,
    0x1.ea4afa2a490dap+0, 0x1.efa1bee615a27p+0, 0x1.f50765b6e4540p+0, 0x1.fa7c1819e90d8p+0,
};

// exp(x) through the table: x = (k ln 2) / 64 + r with |r| < ln 2 / 128, k's low
// six bits the table's entry, the rest the exponent, e^r by its series (r^6 / 720
// < 4e-17 relative): 12 FP64 operations where the general one takes over 20.
// Within 1 ulp.  |x| is held below 2000, so that k fits and an overflow or an
// underflow comes out of the exponent.  (A NaN comes out as 0: see nan_status39.)
struct ExpTab39 {
  const double* tab;  // kExp2_64 in LDS
  __device__ __forceinline__ double operator()(double x) const {
    x = fmin(fmax(x, -2000.0), 2000.0);
    const double magic = 6755399441055744.0;  // 1.5 * 2^52: the sum's low bits are k
    const double t = fma(x, 0x1.71547652b82fep+6, magic);
    const double kd = t - magic;
    const int k = __double2loint(t);
    double r = fma(kd, -0x1.62e42fefa39efp-7, x);
    r = fma(kd, -0x1.abc9e3b39803fp-62, r);
    double q = fma(r, 1.0 / 120.0, 1.0 / 24.0);
    q = fma(q, r, 1.0 / 6.0);
    q = fma(q, r, 0.5);
    q = fma(q, r * r, r);
    const double b = tab[k & 63];
    return ldexp(fma(b, q, b), k >> 6);
  }
};

// alpha's status where a multiplier is a NaN, else 0.  Multiplier 0 stands in
// every exponent: no direction has an equilibrium, the estimate finds nothing to
// sum (1: alpha = 2).  One of the others leaves some directions without: no real
// root (-1), which the step reports.  Settled ahead of the iteration, as the
// exponential above does not carry the NaN (a test of its argument costs each
// exponential three operations) and the shifted lattice's change of basis spreads it.
__device__ __forceinline__ int nan_status39(const double (&lm)[kM39]) {
  bool nan = false;
#pragma unroll
  for (int k = 1; k < kM39; k += 2) nan |= __builtin_isunordered(lm[k], lm[k + 1]);
  return lm[0] != lm[0] ? 1 : nan ? -1 : 0;
}

// exp(-s) for the argument left by a converged Newton's last update: its 13
// entries are below 1e-7 and the monomials of one velocity add up to less than
// 150, so |s| < 1.5e-5 and the next term, s^4 / 24, is below 3e-21
__device__ __forceinline__ double expm_small39(double s) {
  return fma(-s, fma(-s, fma(-s, 1.0 / 6.0, 0.5), 1.0), 1.0);
}

// x^1.5 (NaN for x < 0, as pow gives)
__device__ __forceinline__ double pow15(double x) { return x * sqrt(x); }

// d3q39.h's sutherland39 and therm_cond39 (below 500 K, else that one) with
// pow15: two general powers a node are ~300 operations
__device__ __forceinline__ double sutherland_open39(double T, const Gas39& g, double* dim_mu,
                                                    double* dim_temp) {
  const double const_s = (double)110.15f, temp_ref = (double)273.15f, visc_ref = 1.716e-5;
  const double unit_temp = T * g.t_ref * g.gama;
  const double unit_mu =
      visc_ref * pow15(unit_temp / temp_ref) * ((temp_ref + const_s) / (unit_temp + const_s));
  *dim_mu = unit_mu;
  *dim_temp = unit_temp;
  return unit_mu / g.mu_ref;
}
__device__ __forceinline__ bool therm_cond_open39(double rho, double T, const Gas39& g,
                                                  double* kappa) {
  const double unit_temp = T * g.t_ref * g.gama;
  if (!(unit_temp <= 500.0)) return therm_cond39(rho, T, g, kappa);
  *kappa = 418.1 * (5.9776e-6 * pow15(unit_temp) / (unit_temp + (double)194.4f)) / g.kappa_ref;
  return true;
}

// calculate_alpha.f95:118-289 over the populations f (LDS, full value f_i =
// sf + fref) and the last Newton iteration's equilibrium (LDS, sd).  Returns
// alpha; *st = 0 (root), 1 (alpha = 2), 2 / 3 (clamped low / high), -1 (no
// real root: the reference stops).
template <bool kShifted, typename S>
__device__ __forceinline__ double alpha_open39(const S (*sf)[64], const double (*sd)[64], int t,
                                                   const Ref39& rf, double dim_mu,
                                                   double dim_temp, long long step,
                                                   const Gas39& gs, int* st) {
  const double alpha_hi = 2.125, alpha_start = 1.0e-6;
  const double kb = 1.38064852e-23, pi = 3.1415926535;
  const double mfp = dim_mu / gs.p_ref * sqrt(pi * kb * dim_temp / (2 * gs.molec_weight));
  const double mft = mfp / sqrt(3 * kb * dim_temp / gs.molec_weight);
  const double beta_mfp = gs.dt / (2 * mft + gs.dt);
  double cs1 = 0.0, cs2 = 0.0, cs3 = 0.0;
#pragma unroll 3
  for (int i = 0; i < Q39; ++i) {
    const double f = (double)sf[i][t] + rf.f[i];
    const double d = sd[i][t] - f;
    const double df = f < 0.0 ? fabs(f) : f;
    // x = d / df, df 2x^2/(2+x) and df x^2 over one division: e = df (2 + x)
    // is positive (the equilibrium is), r = 1 / (df e)
    const double e = 2.0 * df + d, r = drcp(df * e), dd = d * d;
    const double x = d * e * r, q2 = dd * e * r;
    cs1 = cs1 + 2.0 * dd * df * r;
    cs2 = cs2 + q2;
    if (x <= 0.0 && x >= -1.0) cs3 = cs3 + q2 * x;
  }
  *st = 0;
  if (fabs(cs3) < 1.24e-16) {
    *st = 1;
    return 2.0;
  }
  double asm_ = (cs2 - sqrt(cs2 * cs2 - 8.0 * cs3 * cs1)) / (2.0 * cs3);
  if (asm_ > alpha_hi) asm_ = alpha_hi - 1.0e-9;
  if (step < gs.startup) asm_ = (asm_ - alpha_start) / (double)gs.startup * (double)step;
  double ft1 = 0, ft2 = 0, ft3 = 0, ft4 = 0, st1 = 0, st2 = 0, third = 0;
#pragma unroll 3
  for (int i = 0; i < Q39; ++i) {
    const double f = (double)sf[i][t] + rf.f[i];
    const double df = f < 0.0 ? fabs(f) : f;
    const double x1 = (sd[i][t] - f) * drcp(df), x2 = x1 * x1, x3 = x2 * x1;
    const double f2 = x2 * df, f3 = x3 * df, f4 = (x2 * x2) * df, f5 = x2 * x3 * df,
                 f6 = (x3 * x3) * df;
    if (x1 <= 0.0 && x1 >= -1.0) {
      ft1 += f3;
      ft2 += f4;
      ft3 += f5;
      ft4 += f6;
    }
    st1 += f2;
    // 2/D1 + 1/D2 + 2/D3 (x1 >= 0 only) and the third-order quotient share
    // one division: r = 1 / (B E), B = D1 D2 D3 or 1
    const double D1 = 4 + asm_ * x1, D2 = 4 + 2 * asm_ * x1, D3 = 4 + 3 * asm_ * x1;
    const bool pos = x1 >= 0.0;
    const double B = pos ? D1 * D2 * D3 : 1.0, E = 60 + 90 * x1 + 36 * x2 + 3 * x3;
    const double r = drcp(B * E);
    if (pos) st2 += f3 * ((2.0 * D2 * D3 + D1 * D3 + 2.0 * D1 * D2) * E * r);
    third = third - (60 * f2 + 60 * f3 + 11 * f4) * B * r;
  }
  const double bm2 = beta_mfp * beta_mfp, b3 = bm2 * beta_mfp;
  const double a2h = alpha_hi * alpha_hi, a3h = a2h * alpha_hi;
  const double first = -bm2 * (ft1 / 6 - alpha_hi * beta_mfp * ft2 / 12 + a2h * bm2 * ft3 / 20 -
                               a3h * b3 * ft4 / 5);
  const double second = st1 / 2 - 2 * asm_ * bm2 * st2 / 15;
  if (fabs(first) < 1.0e-14) {
    *st = 1;
    return 2.0;
  }
  const double na = (-second + sqrt(second * second - 4 * first * third)) / (2 * first);
  if (!(na == na)) {
    *st = -1;
    return 2.0;
  }
  if (na < asm_) {
    *st = 2;
    return asm_;
  }
  if (na > alpha_hi) {
    *st = 3;
    return alpha_hi;
  }
  return na;
}

template <bool kFp32, bool kShifted, bool kTurb, bool kKeepAlpha>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2))) void k39_step_open(
    const void* __restrict__ fA_, const void* __restrict__ gA_, void* __restrict__ fB_,
    void* __restrict__ gB_, double* __restrict__ lmv, double* __restrict__ alpha, Box b, Gas39 gs,
    Ref39 rf, long long step, unsigned long long* __restrict__ stats,
    unsigned* __restrict__ neg_count, unsigned* __restrict__ neg_list) {
  using S = typename std::conditional<kFp32, float, double>::type;
  const S* __restrict__ fA = static_cast<const S*>(fA_);
  const S* __restrict__ gA = static_cast<const S*>(gA_);
  S* __restrict__ fB = static_cast<S*>(fB_);
  S* __restrict__ gB = static_cast<S*>(gB_);
  // staged populations (deviations from the reference equilibrium) in the
  // storage type.  FP64: with g staged as well, two blocks would fill a CU's
  // LDS and leave half its SIMDs idle; g is read again instead
  constexpr bool kStageG = kFp32;
  __shared__ S sf[Q39][64];
  __shared__ S sg[kStageG ? Q39 : 1][64];
  __shared__ double sd[Q39][64];
  __shared__ double etab[64];
  __shared__ signed char nan_ast[64];  // kept here: Newton has no registers for it
  const int t = threadIdx.x;
  etab[t] = kExp2_64[t];
  __syncthreads();
  const unsigned n = (unsigned)b.n;
  const unsigned node = blockIdx.x * 64u + (unsigned)t;
  const bool active = node < n;
  int iters = 0, ast = 0;
  bool noconv = false, kerr = false;
  if (active) {
    const int nx = b.nx, ny = b.ny, nz = b.nz;
    const int x = (int)(node % (unsigned)nx);
    const int y = (int)((node / (unsigned)nx) % (unsigned)ny);
    const int z = (int)(node / ((unsigned)nx * (unsigned)ny));
    auto source = [&](int i) __attribute__((always_inline)) {
      return (unsigned)wrapm(x - cx39<kShifted>(i), nx) +
             (unsigned)nx * ((unsigned)wrapm(y - CY39[i], ny) +
                             (unsigned)ny * (unsigned)wrapm(z - CZ39[i], nz));
    };
    // at one wavefront a SIMD every wait shows: the multipliers are asked for
    // with the populations
    double lm[kM39];
#pragma unroll
    for (int k = 0; k < kM39; ++k) lm[k] = lmv[(size_t)k * n + node];
#pragma unroll
    for (int i = 0; i < Q39; ++i) {
      const unsigned src = source(i);
      sf[i][t] = fA[(size_t)i * n + src];
      if constexpr (kStageG) sg[i][t] = gA[(size_t)i * n + src];
    }
    // g of direction i, from LDS or from registers (read where it is pulled from,
    // for the moments, and again for the collision)
    S gr[kStageG ? 1 : Q39];
    auto g_of = [&](int i) __attribute__((always_inline)) {
      if constexpr (kStageG) return (double)sg[i][t];
      else return (double)gr[i];
    };
    auto read_g = [&]() __attribute__((always_inline)) {
      if constexpr (!kStageG) {
#pragma unroll
        for (int i = 0; i < Q39; ++i) gr[i] = gA[(size_t)i * n + source(i)];
      }
    };
    read_g();
    double rho = 0.0, mx = 0.0, my = 0.0, mz = 0.0, en = 0.0;
#pragma unroll
    for (int i = 0; i < Q39; ++i) {
      const int cx = cx39<kShifted>(i), cy = CY39[i], cz = CZ39[i];
      const double f = (double)sf[i][t] + rf.f[i], g = g_of(i) + rf.g[i];
      const int cm = cx * cx + cy * cy + cz * cz;
      rho += f;
      if (cx) mx = fma((double)cx, f, mx);
      if (cy) my = fma((double)cy, f, my);
      if (cz) mz = fma((double)cz, f, mz);
      en += (double)cm * f + g;
    }
    const double ri = drcp(rho);
    double u[3] = {mx * ri, my * ri, mz * ri};
    const double vm = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    const double T = (en - rho * vm) / (2 * gs.cv * rho);
    const double qf = rho * vm + 5 * rho * T;
    const double tg[kM39] = {rho, rho * u[0], rho * u[1], rho * u[2], rho * (T + u[0] * u[0]),
                             rho * (T + u[1] * u[1]), rho * (T + u[2] * u[2]), rho * u[0] * u[1],
                             rho * u[0] * u[2], rho * u[1] * u[2], qf * u[0], qf * u[1],
                             qf * u[2]};
    if (kTurb) nan_ast[t] = (signed char)nan_status39(lm);
    double dp[kM39];
    // the last iteration's equilibrium stays in LDS for alpha and collision
    const ExpTab39 ex{etab};
    const int it = lm_newton39_groups<kShifted>(
        rho, tg, lm, dp, gs.maxit,
        [&](int i, double e) __attribute__((always_inline)) { sd[i][t] = e; }, ex);
    noconv = it < 0;
    iters = noconv ? gs.maxit : it;
#pragma unroll
    for (int k = 0; k < kM39; ++k) lmv[(size_t)k * n + node] = lm[k];

    // asked for before alpha, which hides the wait; Newton has no registers for it
    __asm__ volatile("" ::: "memory");
    read_g();
    double dim_mu, dim_temp;
    const double mu = sutherland_open39(T, gs, &dim_mu, &dim_temp);
    double al = 2.0;
    if (kTurb) {
      al = alpha_open39<kShifted>(sf, sd, t, rf, dim_mu, dim_temp, step, gs, &ast);
      const int na = nan_ast[t];
      ast = na ? na : ast;
      al = na ? 2.0 : al;
    }
    if (kKeepAlpha) alpha[node] = al;

    // collision: deviation d from the updated multipliers' equilibrium,
    // e_i exp(-(last update) . m_i) with e_i the last iteration's value (d
    // replaces it in LDS), and the signed sums of d and of the g deviation
    const double gT = gs.lead_g * T;
    // Not converged: the update may be large, so the equilibrium itself is
    // formed.  Selects under a uniform branch: with a branch per lane around
    // this block, hipcc (ROCm 7.2) saved registers at its end before it had
    // restored the execution mask, and they were lost.
    if (__any(noconv)) {
#pragma unroll 1
      for (int i = 0; i < Q39; ++i) {
        double s = dp[0];
        const int x = CX39[i], y = CY39[i], z = CZ39[i], c2 = x * x + y * y + z * z;
        const int m[kM39] = {1, x, y, z, x * x, y * y, z * z, x * y, x * z, y * z,
                             x * c2, y * c2, z * c2};
#pragma unroll
        for (int k = 1; k < kM39; ++k) s = fma((double)m[k], dp[k], s);
        sd[i][t] *= noconv ? ex(-s) : 1.0;
      }
#pragma unroll
      for (int k = 0; k < kM39; ++k) dp[k] = noconv ? 0.0 : dp[k];
    }
    Sums39 sum;
    double lq0 = 0, lq1 = 0, lq2 = 0, lqs = 0;
    each39(exponent39(dp), sum, [&](int i, double s) __attribute__((always_inline)) {
      const double feq = expm_small39(s) * sd[i][t];
      const double d = (feq - rf.f[i]) - (double)sf[i][t];
      sd[i][t] = d;
      const double dgi = fma(gT, feq, -rf.g[i]) - g_of(i);
      lqs += dgi;
      if (CX39[i]) lq0 = fma((double)CX39[i], dgi, lq0);
      if (CY39[i]) lq1 = fma((double)CY39[i], dgi, lq1);
      if (CZ39[i]) lq2 = fma((double)CZ39[i], dgi, lq2);
      return d;
    });
    const double eps =
        step < gs.startup ? (((double)step + 1.0) / (double)gs.startup) * gs.eps : gs.eps;
    const double Ti = drcp(T), qs = eps * (1.0 / 6.0) * Ti * Ti * Ti, ql = eps * Ti;
    double kappa = 0.0;
    kerr = !therm_cond_open39(rho, T, gs, &kappa);
    double b1, b2;
    if (step < gs.startup) {
      b1 = gs.init_beta1 + gs.beta1_scale * (double)step;
      b2 = gs.init_beta2 + gs.beta2_scale * (double)step;
    } else {
      b1 = 1.0 / ((ldexp(1.0, gs.lvl + 1) * mu) / (rho * T) + 1.0);
      b2 = 1.0 / ((2.0 * kappa) / (rho * gs.cp * T) + 1.0);
    }
    // f + ab1 (d - qbar) + b2 qbar = f + ab1 d + (b2 - ab1) qbar, g alike
    const double ab1 = al * b1, bq = b2 - ab1;
    Poly39 qb, hq;
    qb = qbar39<kShifted>(sum, u, T, bq * qs);
    {
      // heat flux sum_i (c_i - u) dg_i; c - u = v - (u - shift)
      const double m = bq * ql, ux = kShifted ? u[0] - 1.0 : u[0];
      const double h[3] = {m * fma(-ux, lqs, lq0), m * fma(-u[1], lqs, lq1),
                           m * fma(-u[2], lqs, lq2)};
      hq = linear39<kShifted>(h);
    }
    bool neg = false;
    // the two corrections' values, direction by direction
    each39x2(qb, hq, [&](int i, double qv, double hv) __attribute__((always_inline)) {
      const double d = sd[i][t], s = (double)sf[i][t];
      const double f = s + rf.f[i], g = g_of(i);
      const double dgi = fma(gT, d + f, -rf.g[i]) - g;
      const double fo = s + fma(ab1, d, qv);
      const double go = g + fma(ab1, dgi, hv);
      neg |= fo + rf.f[i] < 0.0;
      fB[(size_t)i * n + node] = (S)fo;
      gB[(size_t)i * n + node] = (S)go;
    });
    if (neg) {
      const unsigned slot = atomicAdd(neg_count, 1u);
      neg_list[slot] = node;
    }
  }
  wave_stats39(stats, active, iters, noconv, ast, kerr);
}

}  // namespace

hipError_t launch_d3q39_step_open(const Box& b, const Step39& a, hipStream_t s) {
  const unsigned blocks = (unsigned)((b.n + 63) / 64);
#define UCLBS_K39O(F, SH, TU, KA)                                                                 \
  hipLaunchKernelGGL((k39_step_open<F, SH, TU, KA>), dim3(blocks), dim3(64), 0, s, a.fin, a.gin,  \
                     a.fout, a.gout, a.lm, a.alpha, b, a.gas, a.ref, (long long)a.step, a.stats,  \
                     a.neg_count, a.neg_list)
#define UCLBS_K39O_KA(F, SH, TU) \
  do { if (a.alpha) UCLBS_K39O(F, SH, TU, true); else UCLBS_K39O(F, SH, TU, false); } while (0)
#define UCLBS_K39O_TU(F, SH) \
  do { if (a.gas.turbulent) UCLBS_K39O_KA(F, SH, true); else UCLBS_K39O_KA(F, SH, false); } while (0)
  if (a.fp32) {
    if (a.shifted) UCLBS_K39O_TU(true, true); else UCLBS_K39O_TU(true, false);
  } else {
    if (a.shifted) UCLBS_K39O_TU(false, true); else UCLBS_K39O_TU(false, false);
  }
#undef UCLBS_K39O_TU
#undef UCLBS_K39O_KA
#undef UCLBS_K39O
  return hipGetLastError();
}

}  // namespace uclbs
