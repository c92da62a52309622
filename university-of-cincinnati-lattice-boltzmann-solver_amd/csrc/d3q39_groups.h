// D3Q39 node update by groups of sign images: the sums and polynomial values of
// the 39 velocities as butterflies, for the levels without boundaries
// (k_d3q39_open.hip).  Same model as d3q39.h; other summation order.
#pragma once
#include "alpha_solve.h"
#include "d3q39.h"

#include <utility>

namespace uclbs {

// The 39 velocities as groups of sign images, in the coordinates v of the plain
// lattice (c = v, on the shifted lattice c = v + (1, 0, 0)): the rest, the eight
// corners (+-1, +-1, +-1), per axis the pairs +-1, +-2, +-3, and per coordinate
// plane the four (+-2, +-2).  A field of the 39 enters every moment through the
// groups' signed sums, and a polynomial in v takes its 39 values from a few
// coefficients a group; both are Walsh-Hadamard butterflies (adds) instead of a
// product per direction and monomial.
__host__ __device__ constexpr int dir39(int x, int y, int z) {
  for (int i = 0; i < 39; ++i)
    if (CX39[i] == x && CY39[i] == y && CZ39[i] == z) return i;
  return -1;
}
// planes xy, xz, yz: their first and second axis
__host__ __device__ constexpr int pax39(int p) { return p == 2 ? 1 : 0; }
__host__ __device__ constexpr int pbx39(int p) { return p == 0 ? 1 : 2; }
struct Dir39 {
  int corner[8];    // component a is -1 where bit a of the index is set
  int axis[3][7];   // k along axis a at [a][k + 3]
  int plane[3][4];  // first / second component -2 where bit 0 / 1 is set
  constexpr Dir39() : corner(), axis(), plane() {
    for (int b = 0; b < 8; ++b) corner[b] = dir39(b & 1 ? -1 : 1, b & 2 ? -1 : 1, b & 4 ? -1 : 1);
    for (int a = 0; a < 3; ++a)
      for (int k = -3; k <= 3; ++k)
        axis[a][k + 3] = dir39(a == 0 ? k : 0, a == 1 ? k : 0, a == 2 ? k : 0);
    for (int p = 0; p < 3; ++p)
      for (int b = 0; b < 4; ++b) {
        int v[3] = {0, 0, 0};
        v[pax39(p)] = b & 1 ? -2 : 2;
        v[pbx39(p)] = b & 2 ? -2 : 2;
        plane[p][b] = dir39(v[0], v[1], v[2]);
      }
  }
};
constexpr Dir39 kDir39{};

template <int kN>
__device__ __forceinline__ void wht39(double (&a)[kN]) {
#pragma unroll
  for (int h = 1; h < kN; h *= 2)
#pragma unroll
    for (int i = 0; i < kN; ++i)
      if (!(i & h)) {
        const double x = a[i], y = a[i + h];
        a[i] = x + y;
        a[i + h] = x - y;
      }
}

// signed sums of a field over the groups: corner sum w[m] and plane sum p[.][m]
// carry the sign of the components in m; s / d: sum and difference of a pair
struct Sums39 {
  double r, w[8], s[3][3], d[3][3], p[3][4];
};

// value polynomial of the groups: rest; on an axis ev k^2 + c0 +- (l k + t k^3);
// corner / plane coefficients by the components whose sign they carry
struct Poly39 {
  double c0, ev[3], l[3], t[3], w[8], p[3][4];
};

// calls fn(i, value) for the 39 directions, group by group; the numbers that fn
// returns are added up in S while the group is in registers
template <class Fn>
__device__ __forceinline__ void each39(const Poly39& q, Sums39& S, Fn&& fn) {
  S.r = fn(0, q.c0);
  {
    double v[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) v[b] = q.w[b];
    wht39<8>(v);
#pragma unroll
    for (int b = 0; b < 8; ++b) v[b] = fn(kDir39.corner[b], v[b]);
    wht39<8>(v);
#pragma unroll
    for (int b = 0; b < 8; ++b) S.w[b] = v[b];
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int k = 1; k <= 3; ++k) {
      const double e = fma((double)(k * k), q.ev[a], q.c0);
      const double o = fma((double)(k * k * k), q.t[a], (double)k * q.l[a]);
      const double x = fn(kDir39.axis[a][k + 3], e + o), y = fn(kDir39.axis[a][3 - k], e - o);
      S.s[a][k - 1] = x + y;
      S.d[a][k - 1] = x - y;
    }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    double v[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) v[b] = q.p[p][b];
    wht39<4>(v);
#pragma unroll
    for (int b = 0; b < 4; ++b) v[b] = fn(kDir39.plane[p][b], v[b]);
    wht39<4>(v);
#pragma unroll
    for (int b = 0; b < 4; ++b) S.p[p][b] = v[b];
  }
}

// two polynomials' values at a time, fn(i, value of q, value of h)
template <class Fn>
__device__ __forceinline__ void each39x2(const Poly39& q, const Poly39& h, Fn&& fn) {
  fn(0, q.c0, h.c0);
  {
    double v[8], w[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) { v[b] = q.w[b]; w[b] = h.w[b]; }
    wht39<8>(v);
    wht39<8>(w);
#pragma unroll
    for (int b = 0; b < 8; ++b) fn(kDir39.corner[b], v[b], w[b]);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int k = 1; k <= 3; ++k) {
      const double e = fma((double)(k * k), q.ev[a], q.c0), f = fma((double)(k * k), h.ev[a], h.c0);
      const double o = fma((double)(k * k * k), q.t[a], (double)k * q.l[a]);
      const double p = fma((double)(k * k * k), h.t[a], (double)k * h.l[a]);
      fn(kDir39.axis[a][3 + k], e + o, f + p);
      fn(kDir39.axis[a][3 - k], e - o, f - p);
    }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    double v[4], w[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) { v[b] = q.p[p][b]; w[b] = h.p[p][b]; }
    wht39<4>(v);
    wht39<4>(w);
#pragma unroll
    for (int b = 0; b < 4; ++b) fn(kDir39.plane[p][b], v[b], w[b]);
  }
}

// axis sums A[a][n] = sum_k k^n (s or d), n = 0..6
struct Axis39 {
  double a[3][7];
  __device__ __forceinline__ explicit Axis39(const Sums39& S) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      a[x][0] = S.s[x][0] + S.s[x][1] + S.s[x][2];
#pragma unroll
      for (int n = 1; n < 7; ++n) {
        const double* v = n & 1 ? S.d[x] : S.s[x];
        a[x][n] = fma((double)(n == 1 ? 3 : n == 2 ? 9 : n == 3 ? 27 : n == 4 ? 81 : n == 5 ? 243 : 729),
                      v[2], fma((double)(1 << n), v[1], v[0]));
      }
    }
  }
};

// moment sum of v_x^p v_y^q v_z^r |v|^(2t) over the field of S
__device__ __forceinline__ double moment39(const Sums39& S, const Axis39& A, int p, int q,
                                                    int r, int t) {
  const int pw[3] = {p, q, r};
  const int bits = (p & 1) | (q & 1) << 1 | (r & 1) << 2;
  double m = t == 0 ? S.w[bits] : t == 1 ? 3.0 * S.w[bits] : 9.0 * S.w[bits];
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) {
    const int a = pax39(pl), b = pbx39(pl), c = 3 - a - b;
    if (pw[c] != 0) continue;
    const double f = (double)(1 << (pw[a] + pw[b] + 3 * t));
    m = fma(f, S.p[pl][(pw[a] & 1) | (pw[b] & 1) << 1], m);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int b = (a + 1) % 3, c = (a + 2) % 3;
    if (pw[b] == 0 && pw[c] == 0) m += A.a[a][pw[a] + 2 * t];
  }
  if (p + q + r + t == 0) m += S.r;
  return m;
}

// powers of the 13 monomials 1, v, v_a^2, v_x v_y, v_x v_z, v_y v_z, v |v|^2
__host__ __device__ constexpr int mpow39(int k, int a) {
  return a == 0 ? (k == 1 || k == 7 || k == 8 || k == 10 ? 1 : k == 4 ? 2 : 0)
       : a == 1 ? (k == 2 || k == 7 || k == 9 || k == 11 ? 1 : k == 5 ? 2 : 0)
       : a == 2 ? (k == 3 || k == 8 || k == 9 || k == 12 ? 1 : k == 6 ? 2 : 0)
                : (k >= 10 ? 1 : 0);
}

// Jacobian entries that hold the same moment: J_kl = sum_i e_i m_k m_l depends
// only on the weights m_k m_l over the 39 directions, and only 57 of the 91
// pairs have distinct ones (x*x = 1*x^2, x^2*y^2 = xy*xy, ...).  rk, rl[p]: the
// first pair of class p, cls[jidx(k, l)] the class of a pair.
struct JClass39 {
  int n;
  signed char rk[91], rl[91], cls[91];
  constexpr JClass39() : n(0), rk(), rl(), cls() {
    for (int k = 0; k < 13; ++k)
      for (int l = 0; l <= k; ++l) {
        int found = -1;
        for (int p = 0; p < n && found < 0; ++p) {
          bool same = true;
          for (int i = 0; i < 39 && same; ++i)
            same = mono39<false>(i, k) * mono39<false>(i, l) ==
                   mono39<false>(i, rk[p]) * mono39<false>(i, rl[p]);
          if (same) found = p;
        }
        if (found < 0) {
          rk[n] = (signed char)k;
          rl[n] = (signed char)l;
          found = n++;
        }
        cls[k * (k + 1) / 2 + l] = (signed char)found;
      }
  }
};
constexpr JClass39 kJClass39{};

// entry q of the packed Jacobian: the moment of its class where it is the
// class's first pair, else that pair's entry (which comes earlier)
template <int kQ>
__device__ __forceinline__ void jacobian_entry39(const Sums39& S, const Axis39& A, double* J) {
  constexpr int c = kJClass39.cls[kQ], k = kJClass39.rk[c], l = kJClass39.rl[c];
  if constexpr (jidx(k, l) == kQ) {
    constexpr int p = mpow39(k, 0) + mpow39(l, 0), q = mpow39(k, 1) + mpow39(l, 1),
                  r = mpow39(k, 2) + mpow39(l, 2), t = mpow39(k, 3) + mpow39(l, 3);
    J[kQ] = moment39(S, A, p, q, r, t);
  } else {
    J[kQ] = J[jidx(k, l)];
  }
}
template <int... kQ>
__device__ __forceinline__ void jacobian39(const Sums39& S, const Axis39& A, double* J,
                                           std::integer_sequence<int, kQ...>) {
  (jacobian_entry39<kQ>(S, A, J), ...);
}

// The shifted lattice's monomials in c = v + (1, 0, 0) span the same space as
// the plain ones in v, and Newton's steps do not depend on the basis: the
// iteration runs in v on both lattices.  Multipliers l (of c) -> p (of v):
template <bool kShifted>
__device__ __forceinline__ void to_plain39(const double* l, double* p) {
#pragma unroll
  for (int k = 0; k < kM39; ++k) p[k] = l[k];
  if constexpr (kShifted) {
    p[0] = (l[0] + l[1]) + (l[4] + l[10]);
    p[1] = fma(3.0, l[10], fma(2.0, l[4], l[1]));
    p[2] = l[2] + (l[7] + l[11]);
    p[3] = l[3] + (l[8] + l[12]);
    p[4] = fma(3.0, l[10], l[4]);
    p[5] = l[5] + l[10];
    p[6] = l[6] + l[10];
    p[7] = fma(2.0, l[11], l[7]);
    p[8] = fma(2.0, l[12], l[8]);
  }
}
template <bool kShifted>
__device__ __forceinline__ void from_plain39(const double* p, double* l) {
#pragma unroll
  for (int k = 0; k < kM39; ++k) l[k] = p[k];
  if constexpr (kShifted) {
    l[8] = fma(-2.0, p[12], p[8]);
    l[7] = fma(-2.0, p[11], p[7]);
    l[6] = p[6] - p[10];
    l[5] = p[5] - p[10];
    l[4] = fma(-3.0, p[10], p[4]);
    l[3] = p[3] - (l[8] + p[12]);
    l[2] = p[2] - (l[7] + p[11]);
    l[1] = fma(-3.0, p[10], fma(-2.0, l[4], p[1]));
    l[0] = p[0] - ((l[1] + l[4]) + p[10]);
  }
}
// moments of the monomials of c -> of v
template <bool kShifted>
__device__ __forceinline__ void moments_plain39(const double* t, double* m) {
#pragma unroll
  for (int k = 0; k < kM39; ++k) m[k] = t[k];
  if constexpr (kShifted) {
    m[1] = t[1] - t[0];
    m[4] = fma(-2.0, t[1], t[4]) + t[0];
    m[7] = t[7] - t[2];
    m[8] = t[8] - t[3];
    m[10] = t[10] - fma(3.0, m[4] + m[1], (t[5] + t[6]) + t[0]);
    m[11] = t[11] - fma(2.0, m[7], t[2]);
    m[12] = t[12] - fma(2.0, m[8], t[3]);
  }
}

// sum_k p_k m_k(v) as a value polynomial
__device__ __forceinline__ Poly39 exponent39(const double* p) {
  Poly39 q;
  q.c0 = p[0];
  double l3[3], l8[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    q.l[a] = p[1 + a];
    q.ev[a] = p[4 + a];
    q.t[a] = p[10 + a];
    l3[a] = fma(3.0, p[10 + a], p[1 + a]);
    l8[a] = fma(16.0, p[10 + a], 2.0 * p[1 + a]);
  }
  q.w[0] = (p[0] + p[4]) + (p[5] + p[6]);
  q.w[1] = l3[0];
  q.w[2] = l3[1];
  q.w[3] = p[7];
  q.w[4] = l3[2];
  q.w[5] = p[8];
  q.w[6] = p[9];
  q.w[7] = 0.0;
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) {
    const int a = pax39(pl), b = pbx39(pl);
    q.p[pl][0] = fma(4.0, p[4 + a] + p[4 + b], p[0]);
    q.p[pl][1] = l8[a];
    q.p[pl][2] = l8[b];
    q.p[pl][3] = 4.0 * p[7 + pl];
  }
  return q;
}

// Newton on the moment constraints; lm in/out, dp = the last update subtracted
// from the multipliers, in the basis of v; sink(i, e) receives each
// iteration's equilibrium (so the caller keeps the last one).  Returns
// iterations, or -1 at the cap.
// An iteration is about 1,700 FP64 operations a node -- 39 exponentials ~600,
// group sums and the 57 moments ~300, L D L^T and the solve ~650 -- where the
// products of each direction with its monomials took 3,400.
template <bool kShifted, class Sink, class Exp>
__device__ __forceinline__ int lm_newton39_groups(double rho, const double tg[kM39], double lm[kM39],
                                           double dp[kM39], int maxit, Sink&& sink, const Exp& ex) {
  double mx = 1.0;
  int it = 0;
  double tp[kM39];
  moments_plain39<kShifted>(tg, tp);
  while (mx > 1.0e-7) {
    if (it >= maxit) return -1;
    ++it;
    double J[kJ39];
    {
      double p[kM39];
      to_plain39<kShifted>(lm, p);
      Sums39 S;
      each39(exponent39(p), S, [&](int i, double x) __attribute__((always_inline)) {
        const double e = rho * ex(x);
        sink(i, e);
        return e;
      });
      const Axis39 A(S);
jacobian39(S, A, J, std::make_integer_sequence<int, kJ39>());
    }
    // residual: current moments (row 0 of J) minus targets
    double r[kM39];
#pragma unroll
    for (int k = 0; k < kM39; ++k) r[k] = J[jidx(k, 0)] - tp[k];
    // L D L^T in place: J[jidx(k,k)] <- D_k, J[jidx(k,l)] <- L_kl (l < k);
    // one reciprocal per pivot
    // v[m] = L_km D_m of the current row: one FMA per update term
    double rD[kM39];
#pragma unroll
    for (int k = 0; k < kM39; ++k) {
      double v[kM39];
#pragma unroll
      for (int l = 0; l < k; ++l) {
        double s = J[jidx(k, l)];
#pragma unroll
        for (int m = 0; m < l; ++m) s = fma(-v[m], J[jidx(l, m)], s);
        v[l] = s;
        J[jidx(k, l)] = s * rD[l];
      }
      double d = J[jidx(k, k)];
#pragma unroll
      for (int m = 0; m < k; ++m) d = fma(-v[m], J[jidx(k, m)], d);
      J[jidx(k, k)] = d;
      rD[k] = drcp(d);
    }
    // solve L y = r, D z = y, L^T delta = z
#pragma unroll
    for (int k = 0; k < kM39; ++k) {
#pragma unroll
      for (int m = 0; m < k; ++m) r[k] -= J[jidx(k, m)] * r[m];
    }
#pragma unroll
    for (int k = 0; k < kM39; ++k) r[k] *= rD[k];
#pragma unroll
    for (int k = kM39 - 1; k >= 0; --k) {
#pragma unroll
      for (int m = k + 1; m < kM39; ++m) r[k] -= J[jidx(m, k)] * r[m];
    }
    double dl[kM39];
    from_plain39<kShifted>(r, dl);
    mx = 0.0;
#pragma unroll
    for (int k = 0; k < kM39; ++k) {
      dp[k] = r[k];
      lm[k] -= dl[k];
      mx = fmax(mx, fabs(dl[k]));
    }
  }
  return it;
}

// qbar of find_q_bar.f95 at the 39 directions, times m: the cubic
// sum_abc Q_abc c_a c_b c_c - 3 T sum_ac Q_aac c_c with Q the central third
// moments of the deviation whose signed sums are S, as a value polynomial in v.
// Q comes from the raw moments in v about u - shift.
template <bool kShifted>
__device__ __forceinline__ Poly39 qbar39(const Sums39& S, const double (&uc)[3], double T, double m) {
  const Axis39 A(S);
  const double u[3] = {kShifted ? uc[0] - 1.0 : uc[0], uc[1], uc[2]};
  const double m0 = moment39(S, A, 0, 0, 0, 0);
  const double m1[3] = {moment39(S, A, 1, 0, 0, 0), moment39(S, A, 0, 1, 0, 0),
                        moment39(S, A, 0, 0, 1, 0)};
  double m2[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = a; b < 3; ++b)
      m2[a][b] = m2[b][a] = moment39(S, A, (a == 0) + (b == 0), (a == 1) + (b == 1),
                                     (a == 2) + (b == 2), 0);
  auto Q = [&](int a, int b, int c) __attribute__((always_inline)) {
    const double m3 = moment39(S, A, (a == 0) + (b == 0) + (c == 0), (a == 1) + (b == 1) + (c == 1),
                               (a == 2) + (b == 2) + (c == 2), 0);
    const double lin = u[a] * u[b] * (m1[c] - u[c] * m0) + u[c] * (u[a] * m1[b] + u[b] * m1[a]);
    return m * (m3 - (u[a] * m2[b][c] + u[b] * m2[a][c] + u[c] * m2[a][b]) + lin);
  };
  const double xxx = Q(0, 0, 0), yyy = Q(1, 1, 1), zzz = Q(2, 2, 2), xxy = Q(0, 0, 1),
               xxz = Q(0, 0, 2), xyy = Q(0, 1, 1), xzz = Q(0, 2, 2), yyz = Q(1, 1, 2),
               yzz = Q(1, 2, 2), xyz = Q(0, 1, 2);
  const double t3 = -3.0 * T;
  // coefficients in c: pure cubes, 3 Q_aab, 6 Q_xyz, and the linear part
  const double xy = 3.0 * xxy, xz = 3.0 * xxz, yx = 3.0 * xyy, zx = 3.0 * xzz, yz = 3.0 * yyz,
               zy = 3.0 * yzz, k = 6.0 * xyz;
  double lx = t3 * (xxx + xyy + xzz), ly = t3 * (xxy + yyy + yzz), lz = t3 * (xxz + yyz + zzz);
  Poly39 q;
  // in v: (v_x + 1)^2 = v_x^2 + 2 v_x + 1 and so on
  double c0 = 0.0, e[3] = {0.0, 0.0, 0.0}, pxy = 0.0, pxz = 0.0, pyz = 0.0;
  if constexpr (kShifted) {
    c0 = xxx + lx;
    lx = fma(3.0, xxx, lx);
    ly += xy;
    lz += xz;
    e[0] = 3.0 * xxx;
    e[1] = yx;
    e[2] = zx;
    pxy = 2.0 * xy;
    pxz = 2.0 * xz;
    pyz = k;
  }
  q.c0 = c0;
  q.ev[0] = e[0]; q.ev[1] = e[1]; q.ev[2] = e[2];
  q.l[0] = lx; q.l[1] = ly; q.l[2] = lz;
  q.t[0] = xxx; q.t[1] = yyy; q.t[2] = zzz;
  q.w[0] = c0 + e[0] + e[1] + e[2];
  q.w[1] = lx + xxx + yx + zx;
  q.w[2] = ly + yyy + xy + zy;
  q.w[4] = lz + zzz + xz + yz;
  q.w[3] = pxy;
  q.w[5] = pxz;
  q.w[6] = pyz;
  q.w[7] = k;
  q.p[0][0] = fma(4.0, e[0] + e[1], c0);
  q.p[0][1] = fma(8.0, xxx + yx, 2.0 * lx);
  q.p[0][2] = fma(8.0, yyy + xy, 2.0 * ly);
  q.p[0][3] = 4.0 * pxy;
  q.p[1][0] = fma(4.0, e[0] + e[2], c0);
  q.p[1][1] = fma(8.0, xxx + zx, 2.0 * lx);
  q.p[1][2] = fma(8.0, zzz + xz, 2.0 * lz);
  q.p[1][3] = 4.0 * pxz;
  q.p[2][0] = fma(4.0, e[1] + e[2], c0);
  q.p[2][1] = fma(8.0, yyy + zy, 2.0 * ly);
  q.p[2][2] = fma(8.0, zzz + yz, 2.0 * lz);
  q.p[2][3] = 4.0 * pyz;
  return q;
}

// sum_a h_a c_a as a value polynomial in v
template <bool kShifted>
__device__ __forceinline__ Poly39 linear39(const double (&h)[3]) {
  Poly39 q;
  q.c0 = kShifted ? h[0] : 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    q.ev[a] = q.t[a] = 0.0;
    q.l[a] = h[a];
    q.p[a][0] = q.c0;
    q.p[a][1] = 2.0 * h[pax39(a)];
    q.p[a][2] = 2.0 * h[pbx39(a)];
    q.p[a][3] = 0.0;
  }
  q.w[0] = q.c0;
  q.w[1] = h[0];
  q.w[2] = h[1];
  q.w[4] = h[2];
  q.w[3] = q.w[5] = q.w[6] = q.w[7] = 0.0;
  return q;
}

}  // namespace uclbs
