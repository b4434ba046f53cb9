// 2D-periodic Ewald lattice sums on gfx950 (ewald.c:260-920) and the e32
// combination into translation coefficients (translations.c:926-1094).
//
// One workgroup per (beta, k, s) "triple": one wave, or several where the triples
// are few; lanes stride over the lattice points (R for the short-range part, K for
// the long-range part), each lane keeps the sigma_{n,m} partial sums in registers,
// and a reduction finishes the triple. The point lists are shared by all triples
// of a batch (one lattice), so they stream from L1/L2. All arithmetic is FP64; the
// short-range integrals use the Faddeeva closed form and the long-range part
// Gamma(1/2 - j, x^2) is evaluated in-kernel (dev_ewald.hpp).
//
// What bounds the sums: FP64 vector instructions (16,000 per triple of LE 7, 433
// R and 2435 K points), and for few triples the length of one wave's walk. Real
// wavenumbers leave nearly everything but the phases real, and both signs of m
// share the phases' steps: 2048 (beta, k) x 3 shifts take 309 us (580 with complex
// arithmetic throughout), one (beta, k) 25 us (138 with one wave per triple); with
// complex k 450 us per 1024 (2190 with continued fractions).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include "dev_ewald.hpp"
#include "dev_specfunc.hpp"
#include "qpms_internal.h"
#include "dev_launch.hpp"

typedef double v2d __attribute__((ext_vector_type(2)));

#define HIPCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) \
  qpms_hip_die(__FILE__, __LINE__, __func__, "HIP error %d (%s) in %s", (int)e_, hipGetErrorString(e_), #x); } while (0)

__constant__ double c_weid[qew::WEID_N];
__constant__ double c_weid_gamma[4][qew::WEID_GN];   // of Gamma(1/2 - J, z), J = 1..4

namespace {

constexpr int cabsi(int a) { return a < 0 ? -a : a; }

// Sum over the wave of each of N values, to tot (LDS): the halves of the wave take
// one half of the values each (one swap of half-waves and one addition for two
// values), then the rows of 16 lanes a half of those, and only N/4 values are
// summed through the 16 lanes. As shuffles of every value these sums were a
// quarter of a short-range triple's instructions.
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return v + __hiloint2double(hi, lo);
}
template <int N>
__device__ __forceinline__ void wave_sums(const double (&v)[N], double *tot) {
  constexpr int H = (N + 1) / 2, Q = (H + 1) / 2;
  const int lane = threadIdx.x & 63;
  double h[2 * Q], q[Q];
#pragma unroll
  for (int i = 0; i < 2 * Q; ++i) {
    const double a = i < H ? v[i] : 0.0, b = i + H < N && i < H ? v[i + H] : 0.0;
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto u = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    h[i] = __hiloint2double((int)u[0], (int)l[0]) + __hiloint2double((int)u[1], (int)l[1]);
  }
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(h[i]), __double2loint(h[i + Q]), false, false);
    const auto u = __builtin_amdgcn_permlane16_swap(__double2hiint(h[i]), __double2hiint(h[i + Q]), false, false);
    q[i] = __hiloint2double((int)u[0], (int)l[0]) + __hiloint2double((int)u[1], (int)l[1]);
    q[i] = dpp_add<0x128>(q[i]);   // row rotated by 8, 4, 2, 1
    q[i] = dpp_add<0x124>(q[i]);
    q[i] = dpp_add<0x122>(q[i]);
    q[i] = dpp_add<0x121>(q[i]);
  }
  const int first = (lane >> 5) * H + ((lane >> 4) & 1) * Q;   // of this row's Q values
  const int end = (lane >> 5) ? N : H;
#pragma unroll
  for (int i = 0; i < Q; ++i)
    if ((lane & 15) == 0 && ((lane >> 4) & 1) * Q + i < H && first + i < end) tot[first + i] = q[i];
}

// The sums of a workgroup's waves (its points' shares) to tot[0]; all threads.
template <int N, int W>
__device__ __forceinline__ void group_sums(const double (&v)[N], double (&tot)[W][N]) {
  const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  wave_sums(v, tot[wave]);
  __syncthreads();
  if (waves > 1) {
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
      double s = tot[0][i];
      for (int w = 1; w < waves; ++w) s += tot[w][i];
      tot[0][i] = s;
    }
    __syncthreads();
  }
}

// Most waves that share a triple: two per SIMD (LE <= 7), or one (LE 9's sums,
// 3D shifts and error estimates need more than half the registers).
template <int LE, bool SMALL = true> constexpr int ew_waves() { return SMALL && LE <= 5 ? 8 : 4; }

// The expansion's coefficients, read again for every point: kept over the points'
// loop they would take 64 registers.
__device__ __forceinline__ const double *weid() {
  const double *a = c_weid;
  asm volatile("" : "+s"(a));
  return a;
}

template <int J>
__device__ __forceinline__ const double *weid_gamma() {
  static_assert(J >= 1 && J <= 4, "expansions for J = 1..4");
  const double *a = c_weid_gamma[J - 1];
  asm volatile("" : "+s"(a));
  return a;
}

__device__ __forceinline__ void acc_add(cplx &acc, double f, cplx e) {
  acc.re = fma(f, e.re, acc.re);
  acc.im = fma(f, e.im, acc.im);
}
__device__ __forceinline__ void acc_add(cplx &acc, cplx f, cplx e) { cfma(acc, f, e); }
__device__ __forceinline__ cplx times(double f, cplx e) { return f * e; }
__device__ __forceinline__ cplx times(cplx f, cplx e) { return f * e; }

// The terms f_n e^{i beta.(R-s)} e^{i m phi} for n + m even: per m the phases of +-m,
// two multiplications for all n.
template <int LE, class V, class Emit>
__device__ __forceinline__ void phase_terms(const V (&f)[LE + 1], cplx phase, cplx e1, Emit emit) {
  cplx up = phase, dn = phase;
#pragma unroll
  for (int m = 0; m <= LE; ++m) {
    if (m > 0) { up = up * e1; dn = dn * conj(e1); }
#pragma unroll
    for (int n = m; n <= LE; n += 2) {
      emit(n, m, f[n], up);
      if (m > 0) emit(n, -m, f[n], dn);
    }
  }
}

// ---------------------------------------------------------------------------
// Short range (ewald.c:742-920):
//   sigma^S_{n,m} = sum_R -i (2/k)^{n+1}/sqrt(pi) |R-s|^n P_n^{|m|}(cos th)
//                   I_n(|R-s|) e^{i beta.(R-s)} e^{i m phi} (-1)^m [m < 0]
// pts: lattice points (x, y, z); the triple's shift s is subtracted.
// XY: all points and s in the plane z = 0: P_n^{|m|}(0) from leg0 and the
// odd n+m coefficients vanish. The factors that do not depend on the point,
// -i (2/k)^{n+1}/sqrt(pi), P_n^{|m|}(0) and the sign of odd negative m, are
// then applied to the sums, and only the (LE+1)(LE+2)/2 coefficients with
// n + m even are accumulated (ev_index).
// ERR: also the error estimate (2^-52 times the sum of |Re| + |Im| of the
// terms).
// ---------------------------------------------------------------------------
template <int LE> constexpr int ev_count() { return (LE + 1) * (LE + 2) / 2; }
__host__ __device__ constexpr int ev_index(int n, int m) { return n * (n + 1) / 2 + (m + n) / 2; }

// KIND: 0 for any k; 1, 2 real and complex k only.
template <int LE, bool XY, bool ERR, int KIND = 0>
__device__ __forceinline__ void short_triple(const double *__restrict__ T /* bx by bz kre kim sx sy sz */, int npts,
                                             const double *__restrict__ pts, double eta,
                                             const double *__restrict__ leg0, int csphase, v2d *__restrict__ out,
                                             double *__restrict__ err) {
  constexpr int NSC = (LE + 1) * (LE + 1);
  constexpr int NA = XY ? ev_count<LE>() : NSC;
  __shared__ double tot[KIND ? 1 : ew_waves<LE, XY && !ERR>()][2 * NA + 1];
  const cplx k = mk(T[3], T[4]);
  const bool kreal = (T[4] == 0.0);
  // -i (2/k)^{n+1} / sqrt(pi): per term (3D shifts) or on the sums (XY)
  const cplx tk = kreal ? mk(2.0 / T[3], 0.0) : 2.0 * cinv(k);
  cplx pre[XY ? 1 : LE + 1];
  if constexpr (!XY) {
    cplx p = tk;
#pragma unroll
    for (int n = 0; n <= LE; ++n) {
      pre[n] = mk(p.im, -p.re) * 0.56418958354775628695;
      p = p * tk;
    }
  }
  cplx acc[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i] = mk(0.0, 0.0);
  double aerr = 0.0;
  // Every short-range term carries exp(-R^2 eta^2 + Re kappa^2), kappa = k / (2 eta):
  // where that exponent is below -746 the factor is exactly 0 in double and
  // so is the term; such points are skipped (the sum is unchanged bit for bit).
  const double kap2re = (T[3] * T[3] - T[4] * T[4]) / (4.0 * eta * eta);
  auto points = [&](auto real) {
  constexpr bool REAL = decltype(real)::value;
  for (int ip = threadIdx.x; ip < npts; ip += blockDim.x) {
    double rx = pts[3 * ip] - T[5], ry = pts[3 * ip + 1] - T[6], rz = pts[3 * ip + 2] - T[7];
    double r = sqrt(rx * rx + ry * ry + rz * rz);
    // R = s: the lattice point coinciding with the particle (the origin for
    // s = 0, translations.c:981-987) carries no short-range term.
    const bool none = r == 0.0 || r * r * eta * eta - kap2re > 746.0;
    if (__all(none)) continue;
    // Else such lanes add zeros (the sums are not held twice): their I_n are zeroed
    // below, and another place makes every other factor finite, which rz / r at r = 0
    // and the phases of a point at infinity are not.
    if (none) { rx = r = 1.0; ry = rz = 0.0; }
    const cplx eb = qew::expi_(T[0] * rx + T[1] * ry + T[2] * rz);
    // e^{i phi}, phi = atan2(ry, rx); on the z axis only m = 0 terms survive
    const double rho = XY ? r : sqrt(rx * rx + ry * ry), irho = qew::rcp_(rho);
    const cplx e1 = (rho != 0.0) ? mk(rx * irho, ry * irho) : mk(1.0, 0.0);
    typename std::conditional<REAL, double, cplx>::type In[LE + 1];
    if constexpr (REAL) qew::sr_integrals_real<LE>(r, k.re, eta, weid(), In);
    else qew::sr_integrals<LE>(r, k, eta, weid(), In);
    {
      double rn = 1.0;   // |R-s|^n I_n
#pragma unroll
      for (int n = 0; n <= LE; ++n) {
        if constexpr (REAL) In[n] = none ? 0.0 : In[n] * rn;
        else In[n] = mk(none ? 0.0 : In[n].re * rn, none ? 0.0 : In[n].im * rn);
        rn *= r;
      }
      if constexpr (XY) {
        phase_terms<LE>(In, eb, e1, [&](int n, int m, auto f, cplx ph) {
          acc_add(acc[ev_index(n, m)], f, ph);
          if (ERR) {
            const cplx b = times(f, ph);
            double tn = 0.56418958354775628695 * cabsd(tk);   // |-i (2/k)^{n+1} / sqrt(pi)|
            for (int i = 0; i < n; ++i) tn *= cabsd(tk);
            aerr += fabs(leg0[n * (n + 1) / 2 + cabsi(m)]) * tn * (fabs(b.re) + fabs(b.im));
          }
        });
      } else {
        double P[qsf::leg_n(LE)];
        const double x = rz / r;
        qsf::legendre_cs<LE>(x, sqrt((1.0 - x) * (1.0 + x)), P);
        cplx em[LE + 1];
        em[0] = mk(1.0, 0.0);
#pragma unroll
        for (int m = 1; m <= LE; ++m) em[m] = em[m - 1] * e1;
#pragma unroll
        for (int n = 0; n <= LE; ++n) {
          cplx base = (pre[n] * In[n]) * eb;
          if (none) base = mk(0.0, 0.0);   // (2/k)^{n+1} may overflow
#pragma unroll
          for (int m = -n; m <= n; ++m) {
            const int am = cabsi(m);
            const double leg = ((csphase == 1) && (am & 1)) ? -P[n * (n + 1) / 2 + am] : P[n * (n + 1) / 2 + am];
            const cplx e = (m >= 0) ? em[am] : conj(em[am]);
            cplx s = (leg * base) * e;
            if (m < 0 && (am & 1)) s = -s;
            acc[n * (n + 1) + m] = acc[n * (n + 1) + m] + s;
            if (ERR) aerr += fabs(s.re) + fabs(s.im);
          }
        }
      }
    }
  }
  };
  if constexpr (KIND != 2) { if (KIND == 1 || kreal) points(std::true_type{}); }
  if constexpr (KIND != 1) { if (KIND == 2 || !kreal) points(std::false_type{}); }
  double v[2 * NA + 1];
#pragma unroll
  for (int i = 0; i < NA; ++i) { v[2 * i] = acc[i].re; v[2 * i + 1] = acc[i].im; }
  v[2 * NA] = ERR ? aerr : 0.0;
  group_sums(v, tot);
  for (int i = threadIdx.x; i < NSC; i += blockDim.x) {
    int n = 0;
    while ((n + 1) * (n + 1) <= i) ++n;
    const int m = i - n * (n + 1), am = m < 0 ? -m : m;
    cplx o;
    if constexpr (XY) {
      o = mk(0.0, 0.0);
      if (!((n + m) & 1)) {
        cplx p = tk;   // (2/k)^{n+1}
        for (int q = 0; q < n; ++q) p = p * tk;
        const int e = ev_index(n, m);
        const double l = leg0[n * (n + 1) / 2 + am], f = (m < 0 && (am & 1)) ? -l : l;
        o = mk(tot[0][2 * e], tot[0][2 * e + 1]) * (mk(p.im, -p.re) * (0.56418958354775628695 * f));
      }
    } else {
      o = mk(tot[0][2 * i], tot[0][2 * i + 1]);
    }
    out[i] = v2d{o.re, o.im};
    if (ERR) err[i] = 2.2204460492503131e-16 * tot[0][2 * NA];
  }
}

// Launch bounds of the kernels by kind of k (one wave per triple): the real ones need
// half the registers without the others' arithmetic beside them, so two waves fit a
// SIMD up to LE 7 (2048 points x 3 shifts, LE 7: 307 us against 498 with one kernel
// for both kinds and one wave per SIMD; few triples are better off with one launch).
#define EW_BOUNDS(LE, KIND, SMALL) \
  __launch_bounds__((KIND ? 64 : 64 * ew_waves<LE, SMALL>()), (KIND && LE <= (KIND == 1 ? 7 : 5) ? 2 : 1))

template <int LE, bool XY, bool ERR, int KIND>
__global__ EW_BOUNDS(LE, KIND, (XY && !ERR)) void k_sigma_short(
    const double *__restrict__ tr, int npts, const double *__restrict__ pts, double eta,
    const double *__restrict__ leg0, int csphase, v2d *__restrict__ out, double *__restrict__ err) {
  constexpr size_t NSC = (LE + 1) * (LE + 1);
  const double *T = tr + 8 * (size_t)blockIdx.x;
  if (KIND && (T[4] == 0.0) != (KIND == 1)) return;
  short_triple<LE, XY, ERR, KIND>(T, npts, pts, eta, leg0, csphase, out + blockIdx.x * NSC,
                            ERR ? err + blockIdx.x * NSC : nullptr);
}

// ---------------------------------------------------------------------------
// Long range, lattice in the xy plane, in-plane shift (ewald.c:286-503):
//   sigma^L_{n,m} = 1/(k^2 A) sum_K e^{i K.s} e^{i m alpha} P_n^{|m|}(0) (-1)^m[m<0]
//     sum_j (|beta+K|/k)^{n-2j} gamma^{2j-1} Gamma(1/2-j, x^2) c_{n,m,j},
//   gamma = clilgamma(|beta+K|/k), x = gamma k / (2 eta).
// c_{n,m,j} = -2 i^{n+1} sqrt(pi) q_{n,|m|,j} (ewald.c:141-145, the s1
// constants), q = (-1)^j a! b! / (j! (a-j)! (b-j)!), a, b = (n -+ |m|)/2: an
// integer. P_n^{|m|}(0) is a dyadic rational, so P_n^{|m|}(0) q_{n,|m|,j} is an
// exact double formed at compile time and the per-term arithmetic has no table
// loads. The factor that remains per coefficient,
//   leg0[n,|m|] / P_n^{|m|}(0) * (-2 sqrt(pi)) i^{n+1}
// (leg0 carries the Condon-Shortley phase the caller chose), is applied to the
// sums (long_out_factor).
// ---------------------------------------------------------------------------
// P_n^{am}(0) without the Condon-Shortley phase (n + am even):
// (-1)^{(n-am)/2} (n+am-1)!! / (n-am)!!
constexpr double ferrers_zero(int n, int am) {
  double num = 1.0, den = 1.0;
  for (int i = n + am - 1; i > 1; i -= 2) num *= i;
  for (int i = n - am; i > 1; i -= 2) den *= i;
  return (((n - am) / 2) & 1) ? -num / den : num / den;
}
// P_n^{am}(0) q_{n,am,j}
constexpr double long_coef_q(int n, int am, int j) {
  const int a = (n - am) / 2, b = (n + am) / 2;
  double f = 1.0;
  for (int i = 0; i < j; ++i) f *= (double)(a - i);              // a! / (a-j)!
  for (int i = 0; i < j; ++i) f = f * (double)(b - i) / (i + 1);  // times C(b, j), exact at each step
  return ferrers_zero(n, am) * ((j & 1) ? -f : f);
}
struct FerrersZero {   // P_n^{am}(0) at n (n + 1) / 2 + am, 1 where it vanishes
  double v[55];
};
constexpr FerrersZero ferrers_zero_table() {
  FerrersZero t{};
  for (int n = 0; n <= 9; ++n)
    for (int am = 0; am <= n; ++am) t.v[n * (n + 1) / 2 + am] = ((n + am) & 1) ? 1.0 : ferrers_zero(n, am);
  return t;
}
__device__ constexpr FerrersZero g_ferrers_zero = ferrers_zero_table();
__device__ __forceinline__ cplx long_out_factor(int n, int am, const double *__restrict__ leg0) {
  const int q = n * (n + 1) / 2 + am;
  const double r = leg0[q] / g_ferrers_zero.v[q] * (-2.0 * 1.7724538509055160273);
  switch ((n + 1) & 3) {   // i^{n+1}
    case 0: return mk(r, 0.0);
    case 1: return mk(0.0, r);
    case 2: return mk(-r, 0.0);
    default: return mk(0.0, -r);
  }
}

// The terms of one K point from rk = |beta+K|/k and gG[j] = gamma^{2j-1}
// Gamma(1/2-j, z), V: double where both are real, else cplx. The m-independent
// products rk^{n-2j} gG[j] are formed once per (n, j), the j sums once per
// (n, |m|) (the sum of -m is that of m, negated for odd |m|), the phases
// phase e^{i m alpha} once per m. emit(e, js, ph): the term of coefficient
// e = ev_index(n, m), n + m even, is js ph (a caller that accumulates needs no
// array of them).
template <int LE, class V, class Emit>
__device__ __forceinline__ void long_terms(V rk, const V (&gG)[LE / 2 + 1], cplx phase, cplx e1, Emit emit) {
  constexpr int JM = LE / 2;
  V rkp[LE + 1], P[LE + 1][JM + 1];
  rkp[0] = rk;
#pragma unroll
  for (int p = 1; p < LE; ++p) rkp[p] = rkp[p - 1] * rk;   // rk^{p+1}
#pragma unroll
  for (int n = 0; n <= LE; ++n)
#pragma unroll
    for (int j = 0; j <= n / 2; ++j) P[n][j] = (n == 2 * j) ? gG[j] : rkp[n == 2 * j ? 0 : n - 2 * j - 1] * gG[j];
  cplx up = phase, dn = phase;
#pragma unroll
  for (int m = 0; m <= LE; ++m) {
    if (m > 0) { up = up * e1; dn = dn * conj(e1); }
#pragma unroll
    for (int n = m; n <= LE; n += 2) {
      V js = P[n][0] * long_coef_q(n, m, 0);
#pragma unroll
      for (int j = 1; j <= (n - m) / 2; ++j) js = js + P[n][j] * long_coef_q(n, m, j);
      emit(ev_index(n, m), js, up);
      if (m > 0) emit(ev_index(n, -m), (m & 1) ? -js : js, dn);
    }
  }
}

// One K point. Nearly all orders of a real wavenumber are evanescent (|beta+K|
// > k): all but the phases is real there, half of the arithmetic.
struct LongPoint {
  double rb;   // |beta+K|
  cplx e1;     // e^{i alpha}, alpha = atan2(by, bx), 0 where beta + K vanishes
};
__device__ __forceinline__ LongPoint long_place(const double *__restrict__ T, double Kx, double Ky) {
  const double bx = Kx + T[0], by = Ky + T[1], rb = sqrt(bx * bx + by * by), irb = qew::rcp_(rb);
  return LongPoint{rb, (rb != 0.0) ? mk(bx * irb, by * irb) : mk(1.0, 0.0)};
}
// Real k: rk = |beta+K|/k and gG[j] = gamma^{2j-1} Gamma(1/2-j, z), z = x^2 =
// (gamma k / (2 eta))^2: 1, 2 (and zeros) where every Gamma underflows, 0 (and
// zeros) where z <= 0.5. The lattice's rings run outwards, so whole waves underflow.
template <int LE>
__device__ __forceinline__ int long_evanescent(double rb, double k, double eta, double &rk, double (&gG)[LE / 2 + 1]) {
  constexpr int JM = LE / 2;
  const double tt = rb / k, kh = k / (2.0 * eta);
  const double g2 = (tt - 1.0) * (tt + 1.0), g = sqrt(g2), x = g * kh, z = x * x;
  const int kind = !(tt >= 1.0 && z > 0.5) ? 0 : z > 740.0 ? 2 : 1;
  rk = kind == 1 ? tt : 1.0;
#pragma unroll
  for (int j = 0; j <= JM; ++j) gG[j] = 0.0;
  if (!__any(kind == 1)) return kind;
  // e^{z} Gamma(1/2 - j, z) from sqrt(pi) erfcx(sqrt z) by the downward
  // recurrence in the order, then e^{-z}
  const double ix = qew::rcp_(x);
  double E[JM + 1];
  qew::gamma_half_scaled<JM>(x, ix, weid(), E);
  double gp = kh * ix * qew::exp_(-z);   // gamma^{2j-1} e^{-z}
#pragma unroll
  for (int j = 0; j <= JM; ++j) {
    gG[j] = kind == 1 ? E[j] * gp : 0.0;
    gp *= g2;
  }
  return kind;
}
// Any order of a real or complex k: false when every Gamma(1/2-j, z) underflows.
template <int LE, bool kreal>
__device__ __forceinline__ bool long_general(double rb, cplx k, double eta, cplx &rk, cplx (&gG)[LE / 2 + 1]) {
  constexpr int JM = LE / 2;
  // gamma, x^2 and the incomplete-gamma branch (ewald.c:384-396)
  cplx gam, z;
  int branch = 0;
  if constexpr (kreal) {
    const double tt = rb / k.re;
    if (tt >= 1.0) {
      gam = mk(sqrt(tt - 1.0) * sqrt(tt + 1.0), 0.0);
      const double x = gam.re * k.re / (2.0 * eta);
      z = mk(x * x, 0.0);
    } else {
      gam = mk(0.0, -(sqrt(1.0 - tt) * sqrt(1.0 + tt)));
      const double x = gam.im * k.re / (2.0 * eta);
      z = mk(-(x * x), -0.0);  // (i x)^2 lies just below the cut
    }
  } else {
    gam = qew::clilgamma(mk(rb, 0.0) / k);
    const cplx x = (gam * k) / (2.0 * eta);
    z = x * x;
    branch = (z.re < 0 && !signbit(z.im)) ? -1 : 0;
  }
  if (z.re > 740.0) return false;
  cplx G[JM + 1];
  if constexpr (kreal) {   // z <= 0.5, or NaN
    qew::gamma_inc_half_real_series<JM>(z, G);
  } else if (z.re > 0.5 && branch == 0) {
    qew::gamma_half_complex<JM>(z, weid_gamma<JM>(), G);
  } else {
#pragma unroll
    for (int j = 0; j <= JM; ++j) G[j] = qew::gamma_inc_half(j, z, branch);
  }
  const cplx g2 = gam * gam;
  cplx gp = cinv(gam);   // gamma^{2j-1}
#pragma unroll
  for (int j = 0; j <= JM; ++j) {
    gG[j] = gp * G[j];
    gp = (j == 0) ? gam : gp * g2;
  }
  rk = kreal ? mk(rb / k.re, 0.0) : mk(rb, 0.0) / k;
  return true;
}

// The waves of a workgroup share the triple's K points, lanes over the points;
// ERR: also the error estimate.
template <int LE, bool ERR, int KIND = 0>
__device__ __forceinline__ void long_triple(const double *__restrict__ T, int npts,
                                            const double *__restrict__ Kp /* x, y */, double eta, double area,
                                            const double *__restrict__ leg0, v2d *__restrict__ out,
                                            double *__restrict__ err) {
  constexpr int NSC = (LE + 1) * (LE + 1), NE = ev_count<LE>();
  __shared__ double tot[KIND ? 1 : ew_waves<LE, !ERR>()][2 * NE + 1];
  const cplx k = mk(T[3], T[4]);
  const bool shifted = T[5] != 0.0 || T[6] != 0.0;   // uniform
  cplx acc[NE];   // the coefficients with n + m even (ev_index); the others vanish
#pragma unroll
  for (int i = 0; i < NE; ++i) acc[i] = mk(0.0, 0.0);
  double aerr = 0.0;
  auto add = [&](int e, auto js, cplx em) {
    acc_add(acc[e], js, em);
    if (ERR) {
      const cplx v = times(js, em);
      aerr += fabs(v.re) + fabs(v.im);
    }
  };
  // Each kind of point where the wave has any, with zeros in the other lanes (sums
  // updated under a lane's condition would be held twice); one loop per kind of k.
  auto points = [&](auto real) {
    constexpr bool REAL = decltype(real)::value;
    for (int ip = threadIdx.x; ip < npts; ip += blockDim.x) {
      double Kx = Kp[2 * ip], Ky = Kp[2 * ip + 1];
      LongPoint at = long_place(T, Kx, Ky);
      double rk, gG[LE / 2 + 1];
      const int ev = REAL ? long_evanescent<LE>(at.rb, k.re, eta, rk, gG) : 0;
      if (REAL && __all(ev == 2)) continue;
      if (REAL && ev == 2) { Kx = Ky = 0.0; at.e1 = mk(1.0, 0.0); }   // zeros times finite phases, at infinity too
      const cplx ph = shifted ? qew::expi_(Kx * T[5] + Ky * T[6]) : mk(1.0, 0.0);
      if (REAL && __any(ev == 1)) long_terms<LE>(rk, gG, ph, at.e1, add);
      if (!REAL || __any(ev == 0)) {
        cplx rc = mk(1.0, 0.0), gc[LE / 2 + 1];
#pragma unroll
        for (int j = 0; j <= LE / 2; ++j) gc[j] = mk(0.0, 0.0);
        const bool live = ev == 0 && long_general<LE, REAL>(at.rb, k, eta, rc, gc);
        if (__any(live)) long_terms<LE>(rc, gc, ph, at.e1, add);
      }
    }
  };
  if constexpr (KIND != 2) { if (KIND == 1 || k.im == 0.0) points(std::true_type{}); }
  if constexpr (KIND != 1) { if (KIND == 2 || k.im != 0.0) points(std::false_type{}); }
  double v[2 * NE + 1];
#pragma unroll
  for (int i = 0; i < NE; ++i) { v[2 * i] = acc[i].re; v[2 * i + 1] = acc[i].im; }
  v[2 * NE] = ERR ? aerr : 0.0;
  group_sums(v, tot);
  const cplx cf = (T[4] == 0.0) ? mk(1.0 / (k.re * k.re * area), 0.0) : cinv((k * k) * area);
  for (int i = threadIdx.x; i < NSC; i += blockDim.x) {
    int n = 0;
    while ((n + 1) * (n + 1) <= i) ++n;
    const int m = i - n * (n + 1);
    cplx o = mk(0.0, 0.0);
    if (!((n + m) & 1)) {
      const int e = ev_index(n, m);
      o = mk(tot[0][2 * e], tot[0][2 * e + 1]) * (cf * long_out_factor(n, m < 0 ? -m : m, leg0));
    }
    out[i] = v2d{o.re, o.im};
    // every out-factor has modulus 2 sqrt(pi) |leg0 / P(0)| = 2 sqrt(pi)
    if (ERR) err[i] = 2.2204460492503131e-16 * tot[0][2 * NE] * (2.0 * 1.7724538509055160273) * cabsd(cf);
  }
}

template <int LE, bool ERR, int KIND>
__global__ EW_BOUNDS(LE, KIND, !ERR) void k_sigma_long(
    const double *__restrict__ tr, int npts, const double *__restrict__ Kp, double eta, double area,
    const double *__restrict__ leg0, v2d *__restrict__ out, double *__restrict__ err) {
  constexpr size_t NSC = (LE + 1) * (LE + 1);
  const double *T = tr + 8 * (size_t)blockIdx.x;
  if (KIND && (T[4] == 0.0) != (KIND == 1)) return;
  long_triple<LE, ERR, KIND>(T, npts, Kp, eta, area, leg0, out + blockIdx.x * NSC,
                       ERR ? err + blockIdx.x * NSC : nullptr);
}

// Both sums of every triple in one launch, in-plane shifts: the long-range ones
// first, they take longer.
template <int LE, int KIND>
__global__ EW_BOUNDS(LE, KIND, true) void k_sigma_both(
    int ntrip, const double *__restrict__ tr, int nR, const double *__restrict__ R, int nK,
    const double *__restrict__ Kp, double eta, double area, const double *__restrict__ leg0, int csphase,
    v2d *__restrict__ ss, v2d *__restrict__ sl) {
  constexpr size_t NSC = (LE + 1) * (LE + 1);
  const int t = blockIdx.x, q = t < ntrip ? t : t - ntrip;
  const double *T = tr + 8 * (size_t)q;
  if (KIND && (T[4] == 0.0) != (KIND == 1)) return;
  if (t < ntrip) long_triple<LE, false, KIND>(T, nK, Kp, eta, area, leg0, sl + q * NSC, nullptr);
  else short_triple<LE, true, false, KIND>(T, nR, R, eta, leg0, csphase, ss + q * NSC, nullptr);
}

// Long range for many shifts sharing (beta, k), as two passes: the terms of
// every K point once (k_long_coef, the same per-point arithmetic as
// k_sigma_long, scaled by 1/(k^2 A)), then per shift the phase sum
// sum_K e^{i K.s} F_K (k_long_shifts).
template <int LE>
__global__ __launch_bounds__(64) void k_long_coef(const double *__restrict__ T, int npts,
                                                   const double *__restrict__ Kp, double eta, double area,
                                                   const double *__restrict__ leg0, v2d *__restrict__ F) {
  constexpr int NE = ev_count<LE>();
  const int ip = blockIdx.x * 64 + threadIdx.x;
  if (ip >= npts) return;
  const cplx k = mk(T[3], T[4]);
  const cplx cf = (T[4] == 0.0) ? mk(1.0 / (k.re * k.re * area), 0.0) : cinv((k * k) * area);
  cplx f[NE];
  const LongPoint at = long_place(T, Kp[2 * ip], Kp[2 * ip + 1]);
  auto keep = [&](int e, auto js, cplx em) { f[e] = times(js, em); };
  bool live = true;
  double rk, gG[LE / 2 + 1];
  const int ev = k.im == 0.0 ? long_evanescent<LE>(at.rb, k.re, eta, rk, gG) : 0;
  if (ev == 1) {
    long_terms<LE>(rk, gG, mk(1.0, 0.0), at.e1, keep);
  } else if (ev == 2) {
    live = false;
  } else {
    cplx rc, gc[LE / 2 + 1];
    live = k.im == 0.0 ? long_general<LE, true>(at.rb, k, eta, rc, gc) : long_general<LE, false>(at.rb, k, eta, rc, gc);
    if (live) long_terms<LE>(rc, gc, mk(1.0, 0.0), at.e1, keep);
  }
#pragma unroll
  for (int n = 0; n <= LE; ++n)
#pragma unroll
    for (int m = -n; m <= n; m += 2) {
      const int e = ev_index(n, m);
      const cplx v = live ? f[e] * (cf * long_out_factor(n, cabsi(m), leg0)) : mk(0.0, 0.0);
      F[(size_t)ip * NE + e] = v2d{v.re, v.im};
    }
}

// The product of the phases (shifts x points) with F (points x coefficients) by
// matrix instructions: 32 shifts and all coefficients per workgroup, whose waves
// share the points, four at a time; every phase is formed once, in the lane that
// feeds it to the matrix instruction, and F is loaded as the other operand. The
// waves' sums are added through LDS, a tile at a time. What bounds it: the matrix
// instructions, 12 for LE 7 beside some 60 vector ones for a phase. One shift per
// thread with F through LDS took 4.9 ms for 4761 shifts (69 particles, LE 7; few
// waves), now 0.35 (0.66 with the points shared by waves and F through scalar loads).
constexpr int LS_W = 8, LS_M = 2;   // waves; tiles of 16 shifts
typedef double v4d __attribute__((ext_vector_type(4)));
template <int LE>
__global__ __launch_bounds__(64 * LS_W) void k_long_shifts(int ntrip, const double *__restrict__ tr, int npts,
                                                           const double *__restrict__ Kp, const v2d *__restrict__ F,
                                                           v2d *__restrict__ out) {
  constexpr int NE = ev_count<LE>(), NSC = (LE + 1) * (LE + 1), NT = (NE + 15) / 16;
  __shared__ double sum[LS_W][8][64];
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s0 = blockIdx.x * 16 * LS_M;
  double sx[LS_M], sy[LS_M];
  v4d re[LS_M][NT], im[LS_M][NT];
#pragma unroll
  for (int i = 0; i < LS_M; ++i) {
    const int t = s0 + 16 * i + lr;
    sx[i] = t < ntrip ? tr[8 * (size_t)t + 5] : 0.0;
    sy[i] = t < ntrip ? tr[8 * (size_t)t + 6] : 0.0;
#pragma unroll
    for (int n = 0; n < NT; ++n) re[i][n] = im[i][n] = v4d{0, 0, 0, 0};
  }
  for (int q0 = 4 * wave; q0 < npts; q0 += 4 * LS_W) {
    const int q = q0 + lk;
    v2d b[NT], K = v2d{0, 0};   // zeros behind the last point and the last coefficient
    if (q < npts) K = v2d{Kp[2 * q], Kp[2 * q + 1]};
#pragma unroll
    for (int n = 0; n < NT; ++n) b[n] = (q < npts && 16 * n + lr < NE) ? F[(size_t)q * NE + 16 * n + lr] : v2d{0, 0};
#pragma unroll
    for (int i = 0; i < LS_M; ++i) {
      const cplx a = qew::expi_(K.x * sx[i] + K.y * sy[i]);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        re[i][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b[n].x, re[i][n], 0, 0, 0);
        im[i][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b[n].y, im[i][n], 0, 0, 0);
        re[i][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b[n].y, re[i][n], 0, 0, 0);
        im[i][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b[n].x, im[i][n], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < LS_M; ++i)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        sum[wave][2 * v][lane] = re[i][n][v];
        sum[wave][2 * v + 1][lane] = im[i][n][v];
      }
      __syncthreads();
      double s = sum[0][wave][lane];   // wave v / 2's row, real or imaginary
      for (int w = 1; w < LS_W; ++w) s += sum[w][wave][lane];
      const int t = s0 + 16 * i + lk + 4 * (wave >> 1), e = 16 * n + lr;
      if (t < ntrip && e < NE) {
        int l = 0;
        while ((l + 1) * (l + 2) / 2 <= e) ++l;
        const int m = 2 * (e - l * (l + 1) / 2) - l;
        reinterpret_cast<double *>(out + (size_t)t * NSC + l * (l + 1) + m)[wave & 1] = s;
      }
    }
  for (int i = threadIdx.x; i < 16 * LS_M * NSC; i += 64 * LS_W) {
    const int t = s0 + i / NSC, y = i % NSC;
    int l = 0;
    while ((l + 1) * (l + 1) <= y) ++l;
    if (t < ntrip && ((y - l * l) & 1)) out[(size_t)t * NSC + y] = v2d{0, 0};   // l + m odd
  }
}

// sigma0 = Gamma(-1/2, -(k/2 eta)^2) P_0^0(0) / (2 sqrt(pi)) (ewald.c:260-273)
__global__ void k_sigma0(int n, const double *__restrict__ kk, double eta, double leg00, v2d *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const cplx k = mk(kk[2 * i], kk[2 * i + 1]);
  cplx z;
  if (k.im == 0.0) {
    const double h = k.re / (2.0 * eta);
    z = mk(-(h * h), -0.0);  // -(k/2eta)^2 with Im = -0 for real k
  } else {
    const cplx h = k / (2.0 * eta);
    z = -(h * h);
  }
  const int branch = (z.re < 0 && !signbit(z.im)) ? -1 : 0;
  const cplx g = qew::gamma_inc_half(1, z, branch);
  const cplx v = g * (leg00 / 2.0 / 1.7724538509055160273);
  out[i] = v2d{v.re, v.im};
}

// ---------------------------------------------------------------------------
// e32 combine (translations.c:1024-1067): per triple, from sigma_total
//   A(y<-yu) = sum_{q<qA} mult_A[q] sigma[y_sc(mu-m, n+nu-2q)]
//   B(y<-yu) = sum_{q<qB'} mult_B[q] sigma[y_sc(mu-m, n+nu-2q+1)]
// qB' = qA (bq_mode 0, the reference's loop bound) or B's own count (mode 1).
// ---------------------------------------------------------------------------
__global__ void k_e32_combine(int ntrip, int nelem, int qslots, int nsc, const v2d *__restrict__ sig,
                              const v2d *__restrict__ mA, const v2d *__restrict__ mB,
                              const unsigned char *__restrict__ qA, const unsigned char *__restrict__ qB,
                              int bq_mode, v2d *__restrict__ A, v2d *__restrict__ B) {
  const int t = blockIdx.y;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntrip || e >= nelem * nelem) return;
  const int y = e / nelem, yu = e % nelem;
  const int n = (int)sqrt((double)y + 1), m = y - n * (n + 1) + 1;
  const int nu = (int)sqrt((double)yu + 1), mu = yu - nu * (nu + 1) + 1;
  const v2d *s = sig + (size_t)t * nsc;
  const int na = qA[e], nb = bq_mode ? qB[e] : qA[e];
  cplx sa = mk(0, 0), sb = mk(0, 0);
  for (int q = 0; q < na; ++q) {
    const int p = n + nu - 2 * q;
    const v2d mq = mA[(size_t)e * qslots + q], sv = s[p * (p + 1) + mu - m];
    cfma(sa, mk(mq.x, mq.y), mk(sv.x, sv.y));
  }
  for (int q = 0; q < nb; ++q) {
    const int p = n + nu - 2 * q + 1;
    const v2d mq = mB[(size_t)e * qslots + q], sv = s[p * (p + 1) + mu - m];
    cfma(sb, mk(mq.x, mq.y), mk(sv.x, sv.y));
  }
  A[(size_t)t * nelem * nelem + e] = v2d{sa.re, sa.im};
  B[(size_t)t * nelem * nelem + e] = v2d{sb.re, sb.im};
}

// sigma_total = short + long (+ sigma0 on y = 0 when flag0[t])
__global__ void k_sigma_total(int ntrip, int nsc, const v2d *__restrict__ ss, const v2d *__restrict__ sl,
                              const v2d *__restrict__ s0, const int *__restrict__ flag0, int parts,
                              v2d *__restrict__ tot) {
  const int t = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntrip || i >= nsc) return;
  v2d v = v2d{0, 0};
  if (parts & 2) v += ss[(size_t)t * nsc + i];
  if (parts & 1) v += sl[(size_t)t * nsc + i];
  if ((parts & 4) && i == 0 && flag0[t]) v += s0[t];
  tot[(size_t)t * nsc + i] = v;
}

}  // namespace

// ---------------------------------------------------------------------------
// Weideman coefficients (host): a_m, m = 1..N, of Weideman's eq. (3.6), from
// the discrete Fourier sum over t_k = L tan(theta_k / 2), theta_k = k pi / M,
// with t^{2J} beside the weight e^{-t^2}: those of w (J = 0), or times
// pi / Gamma(J + 1/2) those of gamma_half_complex.
// ---------------------------------------------------------------------------
static void weideman_coefficients(int N, int J, double *a) {
  const int M = 2 * N, M2 = 2 * M;
  const long double pi = 3.14159265358979323846264338327950288L, L = sqrtl(N / sqrtl(2.0L));
  long double f[4 * 64], scale = 1.0L;
  if (J > 0) {
    scale = sqrtl(pi);
    for (int j = 0; j < J; ++j) scale /= j + 0.5L;
  }
  f[0] = 0.0L;
  for (int k = -M + 1; k <= M - 1; ++k) {
    const long double tt = L * tanl(k * pi / M / 2);
    f[k + M] = expl(-tt * tt) * powl(tt * tt, J) * (L * L + tt * tt);
  }
  for (int m = 1; m <= N; ++m) {
    long double s = 0;
    for (int i = 0; i < M2; ++i) s += f[(i + M) % M2] * cosl(2.0L * pi * (long double)i * m / M2);   // fftshift
    a[m - 1] = (double)(scale * s / M2);
  }
}

static std::once_flag g_weid_once;
static void ensure_weid() {
  std::call_once(g_weid_once, [] {
    double a[qew::WEID_N], g[4][qew::WEID_GN];
    weideman_coefficients(qew::WEID_N, 0, a);
    for (int J = 1; J <= 4; ++J) weideman_coefficients(qew::WEID_GN, J, g[J - 1]);
    HIPCHK(hipMemcpyToSymbol(HIP_SYMBOL(c_weid), a, sizeof a, 0, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpyToSymbol(HIP_SYMBOL(c_weid_gamma), g, sizeof g, 0, hipMemcpyHostToDevice));
  });
}

extern "C" void qh_weideman_coefficients(double *a) { weideman_coefficients(qew::WEID_N, 0, a); }

// Waves per triple: as many as the launch leaves wavefront slots for (2048 of these
// kernels fit on the chip), so that a few triples don't wait for one wave's walk
// through all points: 3 triples 138 us with one wave each, 25 with four (LE 7).
static dim3 triple_threads(int LE, bool small, long blocks) {
  const long most = small && LE <= 5 ? 8 : 4;   // ew_waves
  return dim3((unsigned)(64 * std::max(1L, std::min(most, 2048 / blocks))));
}

extern "C" int qh_launch_sigma_short(int LE, int xy, int ntrip, const double *tr_dev, int npts, const double *pts_dev,
                                     double eta, const double *leg0_dev, int csphase, double *out_dev,
                                     double *err_dev, void *stream) {
  qh_stream(stream);
  ensure_weid();
  if (ntrip <= 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  const dim3 g(ntrip), b = triple_threads(LE, xy && !err_dev, ntrip);
#define QH_SS1(L, X, E, K) QH_LAUNCH((k_sigma_short<L, X, E, K>), g, b, 0, s, tr_dev, npts, pts_dev, eta, leg0_dev, \
      csphase, (v2d *)out_dev, err_dev)
#define QH_SS(L) case L: \
    if (xy) { \
      if (err_dev) QH_SS1(L, true, true, 0); \
      else if (b.x > 64) QH_SS1(L, true, false, 0); \
      else { QH_SS1(L, true, false, 1); QH_SS1(L, true, false, 2); } \
    } else { if (err_dev) QH_SS1(L, false, true, 0); else QH_SS1(L, false, false, 0); } \
    break;
  switch (LE) {
    QH_SS(3) QH_SS(5) QH_SS(7) QH_SS(9)
    default: qpms_hip_die(__FILE__, __LINE__, __func__, "Ewald lMax %d not instantiated (3, 5, 7, 9)", LE);
  }
#undef QH_SS
#undef QH_SS1
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_sigma_long(int LE, int ntrip, const double *tr_dev, int npts, const double *K_dev,
                                    double eta, double area, const double *leg0_dev, double *out_dev,
                                    double *err_dev, void *stream) {
  if (ntrip <= 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  ensure_weid();   // the evanescent orders use the erfcx expansion
  const dim3 g(ntrip), b = triple_threads(LE, !err_dev, ntrip);
#define QH_SL1(L, E, K) QH_LAUNCH((k_sigma_long<L, E, K>), g, b, 0, s, tr_dev, npts, K_dev, eta, area, leg0_dev, \
      (v2d *)out_dev, err_dev)
#define QH_SL(L) case L: \
    if (err_dev) QH_SL1(L, true, 0); \
    else if (b.x > 64) QH_SL1(L, false, 0); \
    else { QH_SL1(L, false, 1); QH_SL1(L, false, 2); } \
    break;
  switch (LE) {
    QH_SL(3) QH_SL(5) QH_SL(7) QH_SL(9)
    default: qpms_hip_die(__FILE__, __LINE__, __func__, "Ewald lMax %d not instantiated (3, 5, 7, 9)", LE);
  }
#undef QH_SL
#undef QH_SL1
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_sigma_both(int LE, int ntrip, const double *tr_dev, int nR, const double *R_dev, int nK,
                                    const double *K_dev, double eta, double area, const double *leg0_dev, int csphase,
                                    double *short_dev, double *long_dev, void *stream) {
  if (ntrip <= 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  ensure_weid();
  // a dispatch takes fewer than 2^26 waves, two for a triple
  constexpr int MOST = 1 << 24;
  if (ntrip > MOST) {
    const size_t nsc2 = 2 * (size_t)(LE + 1) * (LE + 1);
    for (int t = 0; t < ntrip; t += std::min(MOST, ntrip - t))
      qh_launch_sigma_both(LE, std::min(MOST, ntrip - t), tr_dev + 8 * (size_t)t, nR, R_dev, nK, K_dev, eta, area,
                           leg0_dev, csphase, short_dev + nsc2 * t, long_dev + nsc2 * t, stream);
    return 0;
  }
  const dim3 g(2 * (unsigned)ntrip), b = triple_threads(LE, true, 2L * ntrip);
#define QH_SB1(L, K) QH_LAUNCH((k_sigma_both<L, K>), g, b, 0, s, ntrip, tr_dev, nR, R_dev, nK, K_dev, eta, area, \
      leg0_dev, csphase, (v2d *)short_dev, (v2d *)long_dev)
#define QH_SB(L) case L: if (b.x > 64) QH_SB1(L, 0); else { QH_SB1(L, 1); QH_SB1(L, 2); } break;
  switch (LE) {
    QH_SB(3) QH_SB(5) QH_SB(7) QH_SB(9)
    default: qpms_hip_die(__FILE__, __LINE__, __func__, "Ewald lMax %d not instantiated (3, 5, 7, 9)", LE);
  }
#undef QH_SB
#undef QH_SB1
  HIPCHK(hipGetLastError());
  return 0;
}

// Long range for ntrip triples that all share (beta, k) (those of triple 0);
// F: scratch of npts * (LE+1)(LE+2)/2 complex values.
extern "C" size_t qh_sigma_long_shifts_scratch(int LE, int npts) { return (size_t)npts * (LE + 1) * (LE + 2) / 2 * 16; }
extern "C" int qh_launch_sigma_long_shifts(int LE, int ntrip, const double *tr_dev, int npts, const double *K_dev,
                                           double eta, double area, const double *leg0_dev, double *F_dev,
                                           double *out_dev, void *stream) {
  if (ntrip <= 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  ensure_weid();   // the evanescent orders use the erfcx expansion
  const dim3 gc((npts + 63) / 64);
#define QH_LS(L) case L: \
    if (npts > 0) QH_LAUNCH(k_long_coef<L>, gc, dim3(64), 0, s, tr_dev, npts, K_dev, eta, area, leg0_dev, \
                            (v2d *)F_dev); \
    QH_LAUNCH(k_long_shifts<L>, dim3((ntrip + 16 * LS_M - 1) / (16 * LS_M)), dim3(64 * LS_W), 0, s, ntrip, tr_dev, npts, K_dev, (const v2d *)F_dev, \
                       (v2d *)out_dev); break;
  switch (LE) {
    QH_LS(3) QH_LS(5) QH_LS(7) QH_LS(9)
    default: qpms_hip_die(__FILE__, __LINE__, __func__, "Ewald lMax %d not instantiated (3, 5, 7, 9)", LE);
  }
#undef QH_LS
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_sigma0(int n, const double *k_dev, double eta, double leg00, double *out_dev, void *stream) {
  if (n <= 0) return 0;
  QH_LAUNCH(k_sigma0, dim3((n + 63) / 64), dim3(64), 0, (hipStream_t)qh_stream(stream), n, k_dev, eta, leg00,
                     (v2d *)out_dev);
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_sigma_total(int ntrip, int nsc, const double *ss, const double *sl, const double *s0,
                                     const int *flag0, int parts, double *tot, void *stream) {
  if (ntrip <= 0) return 0;
  QH_LAUNCH(k_sigma_total, dim3((nsc + 63) / 64, ntrip), dim3(64), 0, (hipStream_t)qh_stream(stream), ntrip, nsc,
                     (const v2d *)ss, (const v2d *)sl, (const v2d *)s0, flag0, parts, (v2d *)tot);
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_e32_combine(const qh_trans_tables *t, int ntrip, int nsc, const double *sig_dev, int bq_mode,
                                     double *A_dev, double *B_dev, void *stream) {
  if (ntrip <= 0) return 0;
  const int ne = t->nelem;
  QH_LAUNCH(k_e32_combine, dim3((ne * ne + 255) / 256, ntrip), dim3(256), 0, (hipStream_t)qh_stream(stream),
                     ntrip, ne, t->qslots, nsc, (const v2d *)sig_dev, (const v2d *)t->dA, (const v2d *)t->dB, t->dqA,
                     t->dqB, bq_mode, (v2d *)A_dev, (v2d *)B_dev);
  HIPCHK(hipGetLastError());
  return 0;
}
