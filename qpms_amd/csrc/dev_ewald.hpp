// Device special functions for the 2D Ewald sums.
//
//  * Faddeeva w(z) = exp(-z^2) erfc(-iz), Im z >= 0, by Weideman's rational
//    expansion (J.A.C. Weideman, SIAM J. Numer. Anal. 31 (1994) 1497-1518):
//      w(z) = 2 p(Z) / (L - iz)^2 + 1 / (sqrt(pi) (L - iz)),  Z = (L + iz)/(L - iz),
//    p(Z) = sum_{m=1..N} a_m Z^{m-1}, N = 32, L = sqrt(N / sqrt 2). The a_m are
//    computed once on the host (weideman_coefficients) by the discrete Fourier
//    sum of Weideman's eq. (3.6) and live in constant memory.
//    Lower half plane: w(z) = 2 exp(-z^2) - w(-z).
//  * The short-range integrals of the Ewald sum (ewald.c:651-740 evaluates
//    them by adaptive quadrature)
//      I_n(R) = int_eta^inf exp(-R^2 xi^2 + k^2/(4 xi^2)) xi^{2n} d xi,
//    in closed form: with kappa = k/(2 eta), F = exp(-R^2 eta^2 + kappa^2),
//    wp = w(kappa + i R eta), wm = w(-kappa + i R eta)
//      I_0    = F sqrt(pi)/(4R) (wp + wm)
//      I_{-1} = F sqrt(pi)/(2ik) (wp - wm)
//    (Abramowitz & Stegun 7.4.33 with b = -ik/2 and its b-derivative), and the
//    integration-by-parts recurrence
//      I_n = [(2n-1) I_{n-1} - (k^2/2) I_{n-2} + eta^{2n-1} F] / (2 R^2).
//  * Gamma(a, z) for half-integer a = 1/2 - j (ewaldsf.c:44-205 regimes):
//    Legendre continued fraction for Re z >= 0, |z| > 0.5 (DLMF 8.9.2, modified
//    Lentz), otherwise the series Gamma(a) [1 - z^a e^{-z} sum z^k/Gamma(a+k+1)]
//    (DLMF 8.7.3); branch m: Gamma(a, z e^{2 pi i m}) = e^{2 pi i m a} Gamma(a,z)
//    + (1 - e^{2 pi i m a}) Gamma(a) (DLMF 8.2.10).
#pragma once
#include "dev_complex.hpp"

namespace qew {

constexpr int WEID_N = 32;
constexpr int WEID_GN = 40;   // of the incomplete Gamma functions' expansions

// exp, sin and cos, and a reciprocal, for loops whose registers are sums: the
// library's keep their polynomials' coefficients in vector registers over the loop
// (or in scratch, where those do not suffice), evaluate sin and cos apart, and
// carry paths for every argument. Here the coefficients, those of the Taylor
// series, come through scalar loads each time. Errors below 1.5 units in the last
// place.
struct Taylor {
  double s[8], c[9], e[14];   // (-1)^i / (2i+3)!, (-1)^(i+1) / (2i+2)!, 1 / i!
};
constexpr Taylor taylor_table() {
  Taylor t{};
  double f = 1.0;   // i!: exact up to 18!
  for (int i = 0; i <= 19; ++i) {
    if (i > 0) f *= i;
    if (i < 14) t.e[i] = 1.0 / f;
    if (i >= 2 && i % 2 == 0) t.c[i / 2 - 1] = ((i / 2) % 2 ? -1.0 : 1.0) / f;
    if (i >= 3 && i % 2 == 1 && (i - 3) / 2 < 8) t.s[(i - 3) / 2] = ((i - 1) / 2 % 2 ? -1.0 : 1.0) / f;
  }
  return t;
}
#if defined(__HIPCC__)
__device__ constexpr Taylor g_taylor = taylor_table();
__device__ __forceinline__ const Taylor *taylor() {
  const Taylor *t = &g_taylor;
  asm volatile("" : "+s"(t));   // read again each time
  return t;
}

// x != 0, normal and not close to the limits of the range
__device__ __forceinline__ double rcp_(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

__device__ __forceinline__ double exp_(double x) {
  const Taylor *t = taylor();
  x = x > 1100.0 ? 1100.0 : x < -1100.0 ? -1100.0 : x;   // inf and 0 by the scaling; NaN stays
  const double n = rint(x * 1.4426950408889634074);
  double r = fma(n, -6.9314718055994530942e-1, x);        // ln 2 to double
  r = fma(n, -2.3190468138462995584e-17, r);              // and the rest of it
  double p = t->e[13];
#pragma unroll
  for (int i = 12; i >= 0; --i) p = fma(p, r, t->e[i]);
  return ldexp(p, (int)n);
}

// e^{i x}: x - n pi/2 by three fused steps (the first one is exact), |x| < 1e9, else
// the library's. With two steps the smaller part was off by up to 300 units in the last
// place of its own next to multiples of pi/2 (x the double closest to 29 pi/2).
__device__ __forceinline__ cplx expi_(double x) {
  if (__any(!(fabs(x) < 1e9))) return cexpi(x);
  const Taylor *t = taylor();
  const double n = rint(x * 0.63661977236758134308);
  double r = fma(n, -1.5707963267948965580, x);           // pi/2 to double
  r = fma(n, -6.1232339957367660359e-17, r);              // its rest to double
  r = fma(n, 1.4973849048591698329e-33, r);               // and the rest of that
  const double z = r * r;
  double s = t->s[7], c = t->c[8];
#pragma unroll
  for (int i = 6; i >= 0; --i) s = fma(s, z, t->s[i]);
#pragma unroll
  for (int i = 7; i >= 0; --i) c = fma(c, z, t->c[i]);
  s = fma(s * z, r, r);
  c = fma(c, z, 1.0);
  const int q = (int)n;
  const double a = q & 1 ? s : c, b = q & 1 ? c : s;   // cos, sin up to their signs
  return mk((q + 1) & 2 ? -a : a, q & 2 ? -b : b);
}
#endif

QPMS_HD inline cplx cexp2(cplx z) { return cexp_(z); }

// Faddeeva w(z) for Im z >= 0 given the Weideman coefficients a[0..N-1] (a_1..a_N).
QPMS_HD inline cplx faddeeva_uhp(cplx z, const double *a) {
  const double L = 4.7568284600108841;  // sqrt(32 / sqrt(2))
  const cplx iz = mk(-z.im, z.re);
  const cplx den = mk(L, 0.0) - iz;         // L - iz
  const cplx Z = (mk(L, 0.0) + iz) / den;   // (L + iz) / (L - iz)
  cplx p = mk(a[WEID_N - 1], 0.0);
  for (int m = WEID_N - 2; m >= 0; --m) p = p * Z + mk(a[m], 0.0);
  const cplx d2 = den * den;
  return 2.0 * p / d2 + mk(0.56418958354775628695, 0.0) / den;  // 1/sqrt(pi)
}

QPMS_HD inline cplx faddeeva(cplx z, const double *a) {
  if (z.im >= 0.0) return faddeeva_uhp(z, a);
  const cplx mz = -z;
  const cplx e = cexp_(-(z * z));
  return 2.0 * e - faddeeva_uhp(mz, a);
}

// I_n(R), n = 0..NMAX (complex k allowed), into out[0..NMAX].
template <int NMAX>
QPMS_HD inline void sr_integrals(double R, cplx k, double eta, const double *wa, cplx *out) {
  const cplx kap = k / (2.0 * eta);
  const cplx kap2 = kap * kap;
  const double Re = R * eta;
  const cplx F = cexp_(mk(-Re * Re + kap2.re, kap2.im));
  const cplx wp = faddeeva(mk(kap.re, kap.im + Re), wa);
  const cplx wm = faddeeva(mk(-kap.re, -kap.im + Re), wa);
  const double sqpi = 1.7724538509055160273;
  cplx Jm1 = (sqpi * (wp - wm)) / mk(-2.0 * k.im, 2.0 * k.re);  // / (2 i k)
  cplx J0 = (sqpi / (4.0 * R)) * (wp + wm);
  const cplx hk2 = 0.5 * (k * k);
  const double inv2R2 = 1.0 / (2.0 * R * R);
  out[0] = F * J0;
  double etap = eta;  // eta^{2n-1}
  cplx Jn2 = Jm1, Jn1 = J0;
#pragma unroll
  for (int n = 1; n <= NMAX; ++n) {
    const cplx Jn = ((double)(2 * n - 1) * Jn1 - hk2 * Jn2 + mk(etap, 0.0)) * inv2R2;
    out[n] = F * Jn;
    Jn2 = Jn1;
    Jn1 = Jn;
    etap *= eta * eta;
  }
}

// The same for real k, R > 0: with real kappa w(-kappa + i R eta) is the conjugate
// of w(kappa + i R eta), so one expansion serves both and every I_n is real.
#if defined(__HIPCC__)
template <int NMAX>
__device__ __forceinline__ void sr_integrals_real(double R, double k, double eta, const double *wa, double *out) {
  const double kap = k / (2.0 * eta), Re = R * eta;
  const double F = exp_(kap * kap - Re * Re);
  const double L = 4.7568284600108841;                         // sqrt(32 / sqrt(2))
  const double den = L + Re, f = rcp_(den * den + kap * kap);
  const cplx inv = mk(den * f, kap * f);                       // 1 / (L - iz)
  const cplx Z = mk(L - Re, kap) * inv;
  cplx p = mk(wa[WEID_N - 1], 0.0);
#pragma unroll
  for (int m = WEID_N - 2; m >= 0; --m)
    p = mk(fma(p.re, Z.re, fma(-p.im, Z.im, wa[m])), fma(p.re, Z.im, p.im * Z.re));
  const cplx w = inv * (2.0 * (p * inv) + mk(0.56418958354775628695, 0.0));   // 1/sqrt(pi)
  const double sqpi = 1.7724538509055160273;
  const double Jm1 = sqpi * w.im / k, iR = rcp_(R), J0 = (0.5 * sqpi) * iR * w.re;
  const double hk2 = 0.5 * (k * k), inv2R2 = 0.5 * iR * iR;
  out[0] = F * J0;
  double etap = eta;  // eta^{2n-1}
  double Jn2 = Jm1, Jn1 = J0;
#pragma unroll
  for (int n = 1; n <= NMAX; ++n) {
    const double Jn = fma((double)(2 * n - 1), Jn1, fma(-hk2, Jn2, etap)) * inv2R2;
    out[n] = F * Jn;
    Jn2 = Jn1;
    Jn1 = Jn;
    etap *= eta * eta;
  }
}
#endif

// Gamma(a) for a = 1/2 - j.
QPMS_HD inline double gamma_half(int j) {
  double g = 1.7724538509055160273;  // Gamma(1/2)
  for (int i = 0; i < j; ++i) g /= (0.5 - (i + 1));  // Gamma(a-1) = Gamma(a)/(a-1)
  return g;
}

// Principal z^a for half-integer a = 1/2 - j: sqrt(z) * z^{-j}.
QPMS_HD inline cplx cpow_half(cplx z, int j) {
  cplx s = csqrt_(z);
  cplx zi = cinv(z);
  for (int i = 0; i < j; ++i) s = s * zi;
  return s;
}

// Principal log (branch cut on the negative real axis, sign of Im z decides).
QPMS_HD inline cplx clog_(cplx z) { return mk(log(hypot(z.re, z.im)), atan2(z.im, z.re)); }

// Gamma(1/2 - j, z) on branch m (m = 0 principal, m = -1 as used by the
// Ewald sums for Re z < 0 with Im z >= +0).
QPMS_HD inline cplx gamma_inc_half(int j, cplx z, int m) {
  const double a = 0.5 - j;
  cplx val;
  const double az = hypot(z.re, z.im);
  if (z.re >= 0.0 && az > 0.5) {
    // F(a,z) continued fraction (modified Lentz), Gamma = z^{a-1} e^{-z} F.
    const double tiny = 1e-300;
    cplx hn = mk(1.0, 0.0), Cn = mk(1.0 / tiny, 0.0), Dn = mk(1.0, 0.0);
    const cplx zi = cinv(z);
    for (int n = 2; n < 5000; ++n) {
      const cplx an = (n % 2) ? (0.5 * (n - 1)) * zi : (0.5 * n - a) * zi;
      Dn = mk(1.0, 0.0) + an * Dn;
      if (cabs2(Dn) < tiny * tiny) Dn = mk(tiny, 0.0);
      Cn = mk(1.0, 0.0) + an / Cn;
      if (cabs2(Cn) < tiny * tiny) Cn = mk(tiny, 0.0);
      Dn = cinv(Dn);
      const cplx delta = Cn * Dn;
      hn = hn * delta;
      if (cabs2(delta - mk(1.0, 0.0)) < 4.93e-32) break;  // |delta-1| < eps
    }
    const cplx lg = clog_(z);
    const cplx ex = (a - 1.0) * lg - z;
    val = hn * cexp_(ex);
  } else {
    // Gamma(a) [1 - z^a e^{-z} sum_k z^k / Gamma(a+k+1)]
    const double ga = gamma_half(j);
    double gak = ga * a;  // Gamma(a+1)
    cplx zk = mk(1.0, 0.0), sum = mk(0.0, 0.0);
    for (int kk = 0; kk < 200; ++kk) {
      const cplx term = zk / gak;
      sum = sum + term;
      if (kk > 4 && cabs2(term) < 1e-34 * cabs2(sum)) break;
      zk = zk * z;
      gak *= (a + kk + 1);
    }
    const cplx pre = cpow_half(z, j) * cexp_(-z);
    val = ga * (mk(1.0, 0.0) - pre * sum);
  }
  if (m != 0) {
    // e^{2 pi i m a} = (-1)^m for half-integer a
    const double f = (m % 2) ? -1.0 : 1.0;
    val = f * val + mk((1.0 - f) * gamma_half(j), 0.0);
  }
  return val;
}

#if defined(__HIPCC__)
// Gamma(1/2 - j, z), j = 0..J, for real z (Im z = +-0 chooses the side of the cut,
// principal branch) by the series of gamma_inc_half: its sums are real and share
// the reciprocals of the half-integers, one for each power of z.
template <int J>
__device__ __forceinline__ void gamma_inc_half_real_series(cplx z, cplx (&G)[J + 1]) {
  double sum[J + 1], term[J + 1], r[J + 1];
#pragma unroll
  for (int j = 0; j <= J; ++j) {
    term[j] = 1.0 / (gamma_half(j) * (0.5 - j));   // 1 / Gamma(a + 1)
    sum[j] = 0.0;
    r[j] = 1.0 / (1.5 - j);                        // 1 / (a + 1 + k)
  }
  for (int k = 0; k < 200; ++k) {
    bool done = k > 4;
#pragma unroll
    for (int j = 0; j <= J; ++j) {
      sum[j] += term[j];
      done = done && fabs(term[j]) < 1e-17 * fabs(sum[j]);
      term[j] *= z.re * r[j];
    }
    if (done) break;
#pragma unroll
    for (int j = J; j > 0; --j) r[j] = r[j - 1];
    r[0] = rcp_(2.5 + k);
  }
  const double ez = exp_(-z.re);
  const cplx zi = cinv(z);
  cplx p = csqrt_(z);
#pragma unroll
  for (int j = 0; j <= J; ++j) {
    G[j] = gamma_half(j) * (mk(1.0, 0.0) - p * (ez * sum[j]));
    p = p * zi;
  }
}
#endif

#if defined(__HIPCC__)
// Gamma(1/2 - j, z), j = 0..J (J >= 1), for Re z > 0.5 (principal branch). With s = sqrt z
//   e^z Gamma(1/2 - J, z) = s^{1 - 2J} / Gamma(J + 1/2) int e^{-t^2} t^{2J} / (s^2 + t^2) dt
// is w(i s) with t^{2J} beside the weight e^{-t^2}, hence Weideman's expansion with
// coefficients a of that weight, and the lower j follow by the recurrence in the
// direction that keeps relative errors: all within 10 units in the last place for
// 0.5 < Re z, |Im z| < 160. The other direction, from w(i s) itself, loses a factor |z|
// a step (1e-9 at |z| = 300, j = 3). The continued fraction takes 100-340 dependent
// steps of two complex divisions near |z| = 1, for each j.
template <int J>
__device__ __forceinline__ void gamma_half_complex(cplx z, const double *a, cplx (&G)[J + 1]) {
  const double L = 5.3182958969449885;  // sqrt(40 / sqrt(2))
  const cplx s = csqrt_(z), den = mk(L + s.re, s.im);
  const cplx inv = conj(den) * rcp_(cabs2(den)), Z = mk(L - s.re, -s.im) * inv;
  cplx p = mk(a[WEID_GN - 1], 0.0);
#pragma unroll
  for (int m = WEID_GN - 2; m >= 0; --m)
    p = mk(fma(p.re, Z.re, fma(-p.im, Z.im, a[m])), fma(p.re, Z.im, p.im * Z.re));
  cplx E = inv * (2.0 * (p * inv) + mk(1.0, 0.0));
  const cplx ez = exp_(-z.re) * expi_(-z.im), zi = cinv(z);
  cplx za[J + 1];   // z^{1/2 - j}
  za[0] = s;
#pragma unroll
  for (int j = 1; j <= J; ++j) {
    za[j] = za[j - 1] * zi;
    E = E * zi;
  }
  G[J] = E * ez;
#pragma unroll
  for (int j = J; j >= 1; --j) {
    E = za[j] + (0.5 - j) * E;
    G[j - 1] = E * ez;
  }
}
#endif

// Gamma(1/2 - j, x) for real x > 0.5 on the principal branch: the continued
// fraction of gamma_inc_half in real arithmetic (every quantity is real
// there), for the evanescent orders of a real wavenumber. Returns the
// fraction F; Gamma = x^{-1/2-j} e^{-x} F.
QPMS_HD inline double gamma_inc_half_real_cf(int j, double x) {
  const double a = 0.5 - j;
  const double tiny = 1e-300;
  double hn = 1.0, Cn = 1.0 / tiny, Dn = 1.0;
  const double xi = 1.0 / x;
  for (int n = 2; n < 5000; ++n) {
    const double an = (n % 2) ? (0.5 * (n - 1)) * xi : (0.5 * n - a) * xi;
    Dn = 1.0 + an * Dn;
    if (fabs(Dn) < tiny) Dn = tiny;
    Cn = 1.0 + an / Cn;
    if (fabs(Cn) < tiny) Cn = tiny;
    Dn = 1.0 / Dn;
    const double delta = Cn * Dn;
    hn *= delta;
    if (fabs(delta - 1.0) < 2.2204460492503131e-16) break;
  }
  return hn;
}

#if defined(__HIPCC__)
// erfcx(y) = e^{y^2} erfc(y) = w(iy) for real y >= 0: Weideman's expansion on
// the imaginary axis, where Z = (L - y) / (L + y) is real and the whole
// evaluation is real arithmetic (32 FMAs, one division, no exponential).
__device__ __forceinline__ double erfcx_pos(double y, const double *a) {
  const double L = 4.7568284600108841;  // sqrt(32 / sqrt(2))
  const double d = rcp_(L + y);
  const double Z = (L - y) * d;
  double p = a[WEID_N - 1];
  for (int m = WEID_N - 2; m >= 0; --m) p = fma(p, Z, a[m]);
  return d * (2.0 * p * d + 0.56418958354775628695);  // + 1/(sqrt(pi) (L + y))
}

// e^{x} Gamma(1/2 - j, x) for real x > 0 and j = 0..J into E[0..J]:
//   E_0 = sqrt(pi) erfcx(sqrt x)       (Gamma(1/2, x) = sqrt(pi) erfc(sqrt x))
//   E_j = (E_{j-1} - x^{1/2-j}) / (1/2 - j)   (Gamma(a, x) = (Gamma(a+1, x) - x^a e^{-x}) / a).
// The recurrence loses relative digits as x grows (about a factor x / |a| per
// step: 1e-13 at x = 16, j = 4), exactly where Gamma itself carries e^{-x},
// so the absolute error of every term stays at the rounding of O(1) terms;
// for x <= 8 the relative error is below 6e-13 for j <= 4. This replaces a
// continued fraction that needs 100-340 dependent iterations near x = 1.
// Of x the root sx and its reciprocal are given.
template <int J>
__device__ __forceinline__ void gamma_half_scaled(double sx, double isx, const double *a, double (&E)[J + 1]) {
  const double xi = isx * isx;
  E[0] = 1.7724538509055160273 * erfcx_pos(sx, a);
  double xa = sx;  // x^{a}, a = 1/2 - j + 1 at step j
#pragma unroll
  for (int j = 1; j <= J; ++j) {
    xa *= xi;
    E[j] = (E[j - 1] - xa) * (1.0 / (0.5 - j));
  }
}

#endif

QPMS_HD inline double gamma_inc_half_real(int j, double x) {
  return gamma_inc_half_real_cf(j, x) * exp((-0.5 - j) * log(x) - x);
}

// clilgamma(z) (ewald.h:157-170): sqrt(z-1) sqrt(z+1) with the branches
// -pi/2 < arg(z+1) < 3pi/2 and -3pi/2 < arg(z-1) < pi/2.
QPMS_HD inline cplx clilgamma(cplx z) {
  cplx a1 = z - mk(1.0, 0.0), a2 = z + mk(1.0, 0.0);
  a2 = (a2.re < 0 && a2.im <= 0) ? -csqrt_(a2) : csqrt_(a2);
  a1 = (a1.re < 0 && a1.im >= 0) ? -csqrt_(a1) : csqrt_(a1);
  return a1 * a2;
}

}  // namespace qew
