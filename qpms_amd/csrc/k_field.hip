// Incident-field and T-application kernels of the scattering solve.
//
//  k_planewave   regular-VSWF expansion of a plane wave at each particle
//                position (vswf.c:445-530, legendre.c:54-110, normalisation.h:140-210),
//                default normalisation (power-normalised, Condon–Shortley phase).
//                One thread per (particle, y); output in the default basis
//                order: electric block (y = 0..nelem-1), then magnetic block.
//  k_apply_t     f_p = T_{type(p)} a_p for dense nb x nb T per particle type
//                (scatsystem.c:1996-2011 with qpms_apply_tmatrix), one thread
//                per output row.
//  k_cdot        -Re(a^H f) partial sums for the extinction cross-section
//                (misc/finiterectlat-scatter.py:108), one block per batch item.
//  k_scattered_e field of VSWF coefficient vectors at points: per (point,
//                particle) the VSWFs of qpms_vswf_fill_csph (vswf.c:230-288)
//                at k (point - particle), contracted with the particle's
//                coefficients (vswf.c:611-655), turned to cartesian
//                (vectors.h:272-291) and summed over particles
//                (scatsystem.c:2013-2037). One thread per point; when points
//                are few, the waves of a workgroup share 64 points and
//                split the particles.
#include <hip/hip_runtime.h>
#include "dev_ewald.hpp"
#include "dev_specfunc.hpp"
#include "qpms_internal.h"
#include "dev_launch.hpp"

typedef double v2d __attribute__((ext_vector_type(2)));

namespace {

// Ferrers P_l^m (CS phase included) and its x-derivative for l = 1..LMAX,
// m = 0..l, scaled to the spherical-harmonic normalisation divided by
// sqrt(l(l+1)) as qpms_pitau_fill does (legendre.c:89-99).
template <int LMAX>
__device__ void pitau_lm(int l, int m, double x, double st, double &leg, double &pi, double &tau) {
  constexpr double PI_ = 3.14159265358979323846;
  const int am = m < 0 ? -m : m;
  if (fabs(x) == 1.0) {
    // DLMF 14.8.2 limits (legendre.c:65-80)
    leg = 0; pi = 0; tau = 0;
    if (m == 0) leg = ((l & 1) ? x : 1.0) * sqrt((2 * l + 1) / (4 * PI_ * l * (l + 1)));
    if (am == 1) {
      const double fl = 0.25 * sqrt((2 * l + 1) / PI_);
      const double lpar = (l & 1) ? -1.0 : 1.0;
      const double cs = -1.0;
      pi = -((x > 0) ? -1.0 : lpar) * fl * cs;
      tau = ((m > 0) ? 1.0 : -1.0) * ((x > 0) ? 1.0 : lpar) * fl * cs;
    }
    return;
  }
  double P[(LMAX + 1) * (LMAX + 2) / 2];
  qsf::legendre_cs<LMAX>(x, st, P);
  const double Plm = P[qsf::leg_idx(l, am)];
  const double Pl1 = (l - 1 >= am) ? P[qsf::leg_idx(l - 1, am)] : 0.0;
  // (1 - x^2) dP_l^m/dx = (l + m) P_{l-1}^m - l x P_l^m (DLMF 14.10.5)
  const double dP = ((l + am) * Pl1 - l * x * Plm) / ((1.0 - x) * (1.0 + x));
  // sqrt((2l+1)/(4 pi) (l-m)!/(l+m)!) / sqrt(l(l+1))
  double fr = 1.0;
  for (int t = l - am + 1; t <= l + am; ++t) fr *= t;
  double N = sqrt((2 * l + 1) / (4 * PI_ * fr)) / sqrt((double)(l * (l + 1)));
  if (m < 0 && (am & 1)) N = -N;  // negative m: (-1)^m (legendre.c:25-33)
  leg = N * Plm;
  const double legder = N * dP;
  pi = m / st * leg;
  tau = -st * legder;
}

template <int LMAX>
__global__ void k_planewave(int npart, const double *__restrict__ pos, double kx, double ky, double kz,
                            const double *__restrict__ Ecart, v2d *__restrict__ out, long ld) {
  constexpr int NE = LMAX * (LMAX + 2);
  constexpr double PI_ = 3.14159265358979323846;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npart * NE) return;
  const int p = t / NE, y = t % NE;
  int l = 1;
  while ((l + 1) * (l + 1) - 1 <= y) ++l;  // y = l(l+1) + m - 1, |m| <= l
  const int m = y - l * (l + 1) + 1;
  // direction of Re k (cart2sph, vectors.h:134-140)
  const double kr = sqrt(kx * kx + ky * ky + kz * kz);
  const double theta = kr != 0.0 ? acos(kz / kr) : PI_ / 2;
  const double phi = atan2(ky, kx);
  const double ct = cos(theta), st = sin(theta), cf = cos(phi), sf = sin(phi);
  double leg, pi, tau;
  pitau_lm<LMAX>(l, m, ct, st, leg, pi, tau);
  // E in the local geographic basis (ccart2csphvec, vectors.h:306-327)
  const cplx Ex = mk(Ecart[0], Ecart[1]), Ey = mk(Ecart[2], Ecart[3]), Ez = mk(Ecart[4], Ecart[5]);
  const cplx Et = (ct * cf) * Ex + (ct * sf) * Ey + (-st) * Ez;
  const cplx Ef = (-sf) * Ex + cf * Ey;
  // dual waves: e^{-i m phi}, derivative/m = -i e^{-i m phi} (normalisation.h:140-205)
  const cplx eimf = cexpi(-m * phi);
  const cplx deimf = (m == 0) ? mk(0.0, 0.0) : mk(eimf.im, -eimf.re);
  // A1 = (0, pi d, -tau e), A2 = (0, tau e, pi d) (vswf.c:347-381)
  const cplx dot1 = (pi * deimf) * Et + (-tau * eimf) * Ef;
  const cplx dot2 = (tau * eimf) * Et + (pi * deimf) * Ef;
  // 4 pi i^l and -4 pi i^(l+1) (vswf.c:455-462)
  const cplx il = ((l & 3) == 0) ? mk(1, 0) : ((l & 3) == 1) ? mk(0, 1) : ((l & 3) == 2) ? mk(-1, 0) : mk(0, -1);
  const cplx il1 = mk(-il.im, il.re);
  const cplx mg = (4 * PI_) * il * dot1;
  const cplx el = (-4 * PI_) * il1 * dot2;
  // phase e^{i k.r} of the expansion point (vswf.c:486-488)
  const double ph = kx * pos[3 * p] + ky * pos[3 * p + 1] + kz * pos[3 * p + 2];
  const cplx f = cexpi(ph);
  const cplx e1 = el * f, m1 = mg * f;
  out[(size_t)p * ld + y] = v2d{e1.re, e1.im};
  out[(size_t)p * ld + NE + y] = v2d{m1.re, m1.im};
}

// out[p] = T[ttype[p]] a[p], T row-major nb x nb per type.
__global__ void k_apply_t(int npart, int nb, const int *__restrict__ ttype, const v2d *__restrict__ T,
                          const v2d *__restrict__ a, v2d *__restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npart * nb) return;
  const int p = t / nb, r = t % nb;
  const v2d *Tr = T + ((size_t)ttype[p] * nb + r) * nb;
  const v2d *ap = a + (size_t)p * nb;
  double sr = 0, si = 0;
  for (int c = 0; c < nb; ++c) {
    const v2d x = Tr[c], v = ap[c];
    sr += x.x * v.x - x.y * v.y;
    si += x.x * v.y + x.y * v.x;
  }
  out[(size_t)p * nb + r] = v2d{sr, si};
}

// partial[b] = -Re(sum_i conj(a_i) f_i) over n entries of batch item b.
__global__ void k_neg_re_cdot(long n, const v2d *__restrict__ a, long sa, const v2d *__restrict__ f, long sf,
                              double *__restrict__ out) {
  __shared__ double red[256];
  const v2d *ab = a + (size_t)blockIdx.x * sa, *fb = f + (size_t)blockIdx.x * sf;
  double s = 0;
  for (long i = threadIdx.x; i < n; i += blockDim.x) {
    const v2d x = ab[i], y = fb[i];
    s += x.x * y.x + x.y * y.y;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = -red[0];
}


// Which radial functions: any kind, at the origin too (regular waves); h_l of
// complex and of real k r, formed directly at every argument (the outgoing field's
// case; the origin is then a singular point, NaN).
enum { RADIAL_ANY, RADIAL_HANKEL, RADIAL_HANKEL_REAL };

// One particle's field at offset (dx, dy, dz) from it, added to E (cartesian).
// c: the particle's 2 NE coefficients (electric block, then magnetic);
// parity: multiply electric coefficients by (-1)^(l+1), magnetic by (-1)^l.
//
// The angular functions of m >= 1 come from Q_l^m = P_l^m / sin(theta), which has
// the recurrence of P_l^m and is finite on the axis:
//   leg = N sin Q_l^m, pi = N m Q_l^m, tau = N (l cos Q_l^m - (l+m) Q_{l-1}^m),
//   m = 0: tau = N P_l^1
// (DLMF 14.10.5), so nothing is divided by sin(theta) and the poles' limits
// (legendre.c:65-80) come out by themselves. +-m share them: with a = c_m e^{i m
// phi}, b = (-1)^m c_{-m} e^{-i m phi} the sums take leg (a + b), tau (a + b) and
// pi (a - b).
template <int LMAX, int RADIAL>
__device__ __forceinline__ void field_of_particle(double dx, double dy, double dz, cplx k, int kind,
                                                  const v2d *__restrict__ c, bool parity, cplx *E) {
  constexpr int NE = LMAX * (LMAX + 2);
  constexpr double PI_ = 3.14159265358979323846;
  // direction cosines of cart2sph's (theta, phi) (vectors.h:134-140): theta =
  // pi/2 at r = 0; phi = 0 or pi on the z axis
  const double rho2 = dx * dx + dy * dy, r = sqrt(rho2 + dz * dz), rho = sqrt(rho2);
  const double ir = qew::rcp_(r), irho = qew::rcp_(rho);
  const double ct = r != 0.0 ? dz * ir : cos(PI_ / 2), st = r != 0.0 ? rho * ir : 1.0;
  const double cf = rho != 0.0 ? dx * irho : copysign(1.0, dx), sf = rho != 0.0 ? dy * irho : 0.0;
  cplx z[LMAX + 1], krinv;
  const cplx kr = k * r;
  const bool origin = (kr.re == 0.0 && kr.im == 0.0);
  if constexpr (RADIAL == RADIAL_HANKEL_REAL) {
    const double sg = (kind == 3) ? 1.0 : -1.0, zi = qew::rcp_(kr.re);   // NaN at the origin
    const cplx e = qew::expi_(sg * kr.re);
    z[0] = mk(sg * zi * e.im, -sg * zi * e.re);                          // -+i e^{+-ix}/x
    z[1] = -(zi * zi) * (e * mk(kr.re, sg));
#pragma unroll
    for (int l = 1; l < LMAX; ++l) {
      const double f = (double)(2 * l + 1) * zi;
      z[l + 1] = mk(fma(f, z[l].re, -z[l - 1].re), fma(f, z[l].im, -z[l - 1].im));
    }
    krinv = mk(zi, 0.0);
  } else {
    if (RADIAL == RADIAL_HANKEL) {
      if (origin) {   // h_l is singular at the origin (as sph_bessel_fill gives it)
#pragma unroll
        for (int l = 0; l <= LMAX; ++l) z[l] = mk(NAN, NAN);
      } else {
        qsf::sph_hankel_direct<LMAX>(kind, kr, z);
      }
    } else {
      qsf::sph_bessel_fill<LMAX>(kind, kr, z);
    }
    krinv = origin ? mk(0.0, 0.0) : cinv(kr);
  }
  double P[LMAX + 1], Q[LMAX + 1][LMAX + 1];   // P_l^0; Q_l^m
  P[0] = 1.0;
  P[1] = ct;
#pragma unroll
  for (int l = 2; l <= LMAX; ++l) P[l] = ((2 * l - 1) / (double)l) * (ct * P[l - 1]) - ((l - 1) / (double)l) * P[l - 2];
  cplx em[LMAX + 1];   // e^{i m phi}
  em[0] = mk(1.0, 0.0);
#pragma unroll
  for (int m = 1; m <= LMAX; ++m) {
    em[m] = m == 1 ? mk(cf, sf) : em[m - 1] * mk(cf, sf);
    Q[m][m] = m == 1 ? -1.0 : (-(2 * m - 1) * st) * Q[m - 1][m - 1];
    Q[m - 1][m] = 0.0;
#pragma unroll
    for (int l = m + 1; l <= LMAX; ++l)
      Q[l][m] = ((2 * l - 1) / (double)(l - m)) * (ct * Q[l - 1][m]) - ((l + m - 1) / (double)(l - m)) * Q[l - 2 < m ? m - 1 : l - 2][m];
  }
  cplx Er = mk(0.0, 0.0), Et = mk(0.0, 0.0), Ef = mk(0.0, 0.0);
#pragma unroll
  for (int l = 1; l <= LMAX; ++l) {
    // z_l / kr (1/3 for the regular l = 1 wave at the origin) and z_{l-1} - l z_l / kr
    cplx besfac, zl = z[l];
    if constexpr (RADIAL == RADIAL_HANKEL_REAL) besfac = krinv.re * z[l];
    else besfac = origin ? mk(l == 1 ? 1.0 / 3.0 : 0.0, 0.0) : z[l] * krinv;
    cplx besder = z[l - 1] - (double)l * besfac;
    if (parity) {   // uniform; electric: (-1)^(l+1), magnetic: (-1)^l
      if (l & 1) zl = -zl;
      else besfac = -besfac, besder = -besder;
    }
    // angular sums of degree l; the radial factors multiply them once per l:
    // N = (l(l+1) leg z/kr e, tau besder e, pi besder i e), M = (0, pi z i e, -tau z e)
    const int y0 = l * (l + 1) - 1;
    const double n0 = sqrt((2 * l + 1) / (4 * PI_)) / sqrt((double)(l * (l + 1)));
    const cplx c0 = mk(c[y0].x, c[y0].y), d0 = mk(c[NE + y0].x, c[NE + y0].y);
    const double leg0 = n0 * P[l], tau0 = n0 * (st * Q[l][1]);
    cplx sLegN = leg0 * c0, sTauN = tau0 * c0, sPiN = mk(0.0, 0.0), sPiM = mk(0.0, 0.0), sTauM = tau0 * d0;
#pragma unroll
    for (int m = 1; m <= l; ++m) {
      double fr = 1.0;
#pragma unroll
      for (int t = l - m + 1; t <= l + m; ++t) fr *= t;
      const double nlm = sqrt((2 * l + 1) / (4 * PI_ * fr)) / sqrt((double)(l * (l + 1)));
      const double q = nlm * Q[l][m], leg = st * q, pi = m * q;
      const double tau = m == l ? (l * ct) * q : fma(l * ct, q, (-(l + m) * nlm) * Q[l - 1][m]);
      const v2d cp = c[y0 + m], cn = c[y0 - m], dp = c[NE + y0 + m], dn = c[NE + y0 - m];
      const cplx e = em[m], a = mk(cp.x, cp.y) * e, b = mk(cn.x, cn.y) * conj(e), f = mk(dp.x, dp.y) * e,
                 g = mk(dn.x, dn.y) * conj(e);
      const cplx ps = (m & 1) ? a - b : a + b, pd = (m & 1) ? a + b : a - b;
      const cplx qs = (m & 1) ? f - g : f + g, qd = (m & 1) ? f + g : f - g;
      sLegN = sLegN + leg * ps;
      sTauN = sTauN + tau * ps;
      sPiN = sPiN + pi * pd;
      sPiM = sPiM + pi * qd;
      sTauM = sTauM + tau * qs;
    }
    const cplx zs = zl * sPiM, bs = besder * sPiN;
    Er = Er + (double)(l * (l + 1)) * (besfac * sLegN);
    Et = Et + besder * sTauN + mk(-zs.im, zs.re);
    Ef = Ef + mk(-bs.im, bs.re) - zl * sTauM;
  }
  E[0] = E[0] + (st * cf) * Er + (ct * cf) * Et - sf * Ef;
  E[1] = E[1] + (st * sf) * Er + (ct * sf) * Et + cf * Ef;
  E[2] = E[2] + ct * Er - st * Et;
}

// One thread per point, 64 points per wave; the S waves of a group share
// their 64 points and split the particles (wave w of the group takes
// p = w, w + S, ...), so a particle's position and coefficients are the same
// for the whole wave (scalar loads, read once per wave instead of once per
// lane) and points too few to fill the device still give S times as many
// waves. The S partial fields of a point are added in LDS in slice order
// (deterministic).
//
// What bounds it: FP64 vector instructions, 565 per wave and particle for lMax 3
// and real k (84 % of their issue rate at 65,536 points and 1024 particles: 1.12
// ms). With P_l^m divided by sin(theta) per (l, m), the poles apart, each sign of m
// by itself and the library's sin, cos and exp it took 1300 and 2.80 ms.
template <int LMAX, int S, int RADIAL>
__global__ __launch_bounds__((S > 4 ? 64 * S : 256), (LMAX <= 3 ? 2 : 1)) void k_scattered_e(int npts, const double *__restrict__ where, int npart,
                                                     const double *__restrict__ pos, double k_re, double k_im,
                                                     int kind, const v2d *__restrict__ cvf, int parity,
                                                     v2d *__restrict__ out) {
  constexpr int NB = 2 * LMAX * (LMAX + 2), W = S > 4 ? S : 4, G = W / S;   // waves, point groups per workgroup
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int slice = __builtin_amdgcn_readfirstlane(wave % S), grp = wave / S;
  const int t = (blockIdx.x * G + grp) * 64 + lane;
  const bool live = t < npts;
  const cplx k = mk(k_re, k_im);
  cplx E[3] = {mk(0.0, 0.0), mk(0.0, 0.0), mk(0.0, 0.0)};
  if (live) {
    const double wx = where[3 * t], wy = where[3 * t + 1], wz = where[3 * t + 2];
    for (int p = slice; p < npart; p += S)
      field_of_particle<LMAX, RADIAL>(wx - pos[3 * p], wy - pos[3 * p + 1], wz - pos[3 * p + 2], k, kind,
                                      cvf + (size_t)p * NB, parity != 0, E);
  }
  if (S > 1) {
    __shared__ double red[W][6][64];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      red[wave][2 * q][lane] = E[q].re;
      red[wave][2 * q + 1][lane] = E[q].im;
    }
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int w = 1; w < S; ++w)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        E[q].re += red[wave + w][2 * q][lane];
        E[q].im += red[wave + w][2 * q + 1][lane];
      }
  }
  if (!live) return;
#pragma unroll
  for (int q = 0; q < 3; ++q) out[3 * (size_t)t + q] = v2d{E[q].re, E[q].im};
}

}  // namespace

#define HIPCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) \
  qpms_hip_die(__FILE__, __LINE__, __func__, "HIP error %d (%s) in %s", (int)e_, hipGetErrorString(e_), #x); } while (0)

extern "C" int qh_launch_planewave(int lMax, size_t npart, const double *pos_dev, const double kvec[3],
                                   const double *E_dev, double *out_dev, long ld, void *stream) {
  if (npart == 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  const int ne = lMax * (lMax + 2);
  const dim3 grid((unsigned)((npart * ne + 255) / 256)), block(256);
  v2d *o = (v2d *)out_dev;
  switch (lMax) {
    case 1: QH_LAUNCH(k_planewave<1>, grid, block, 0, s, (int)npart, pos_dev, kvec[0], kvec[1], kvec[2], E_dev, o, ld); break;
    case 2: QH_LAUNCH(k_planewave<2>, grid, block, 0, s, (int)npart, pos_dev, kvec[0], kvec[1], kvec[2], E_dev, o, ld); break;
    case 3: QH_LAUNCH(k_planewave<3>, grid, block, 0, s, (int)npart, pos_dev, kvec[0], kvec[1], kvec[2], E_dev, o, ld); break;
    case 4: QH_LAUNCH(k_planewave<4>, grid, block, 0, s, (int)npart, pos_dev, kvec[0], kvec[1], kvec[2], E_dev, o, ld); break;
    default: qpms_hip_die(__FILE__, __LINE__, __func__, "lMax %d not instantiated (1..4)", lMax);
  }
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_apply_t(size_t npart, int nb, const int *ttype_dev, const double *T_dev, const double *a_dev,
                                 double *out_dev, void *stream) {
  if (npart == 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  const dim3 grid((unsigned)((npart * nb + 255) / 256)), block(256);
  QH_LAUNCH(k_apply_t, grid, block, 0, s, (int)npart, nb, ttype_dev, (const v2d *)T_dev,
                     (const v2d *)a_dev, (v2d *)out_dev);
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int qh_launch_neg_re_cdot(int batch, long n, const double *a_dev, long sa, const double *f_dev, long sf,
                                     double *out_dev, void *stream) {
  if (batch == 0) return 0;
  hipStream_t s = (hipStream_t)qh_stream(stream);
  QH_LAUNCH(k_neg_re_cdot, dim3(batch), dim3(256), 0, s, n, (const v2d *)a_dev, sa, (const v2d *)f_dev, sf,
                     out_dev);
  HIPCHK(hipGetLastError());
  return 0;
}

// Points at where[3 npts], particles at pos[3 npart], coefficients cvf[npart][2 nelem(lMax)];
// out[3 npts] complex. parity != 0 multiplies electric coefficients by (-1)^(l+1)
// and magnetic ones by (-1)^l first.
extern "C" int qh_launch_scattered_e(int lMax, size_t npts, const double *where_dev, size_t npart,
                                     const double *pos_dev, double k_re, double k_im, int kind,
                                     const double *cvf_dev, int parity, double *out_dev, void *stream) {
  if (npts == 0) return 0;
  if (npts > (size_t)INT32_MAX || npart > (size_t)INT32_MAX)
    qpms_hip_die(__FILE__, __LINE__, __func__, "too many points (%zu) or particles (%zu)", npts, npart);
  hipStream_t s = (hipStream_t)qh_stream(stream);
  // points too few to fill the device one thread each (fewer than 262,144,
  // 4096 waves): the particles split over 4 waves per 64 points; over 8 where even
  // their workgroups are fewer than the CUs (16,384: 1000 particles of lMax 3 at
  // 10,000 points 325 us against 395 with 4; at 65,536, where 8 waves of a workgroup
  // leave a third of the registers unused, 4 win: 1.12 against 1.20 ms)
  const int S = (npart < 4 || npts >= 262144) ? 1 : npts < 16384 ? 8 : 4, W = S > 4 ? S : 4;
  const int radial = kind < 3 ? RADIAL_ANY : k_im == 0.0 ? RADIAL_HANKEL_REAL : RADIAL_HANKEL;
  const dim3 grid((unsigned)((npts + 64 * (W / S) - 1) / (64 * (W / S)))), block(64 * W);
  const v2d *c = (const v2d *)cvf_dev;
  v2d *o = (v2d *)out_dev;
#define QH_SCE1(LM, SL, H) \
  QH_LAUNCH((k_scattered_e<LM, SL, H>), grid, block, 0, s, (int)npts, where_dev, (int)npart, pos_dev, k_re, \
                     k_im, kind, c, parity, o)
#define QH_SCE2(LM, SL)                                                    \
  do {                                                                     \
    if (radial == RADIAL_HANKEL_REAL) QH_SCE1(LM, SL, RADIAL_HANKEL_REAL); \
    else if (radial == RADIAL_HANKEL) QH_SCE1(LM, SL, RADIAL_HANKEL);      \
    else QH_SCE1(LM, SL, RADIAL_ANY);                                      \
  } while (0)
#define QH_SCE(LM)               \
  do {                           \
    if (S == 8) QH_SCE2(LM, 8);  \
    else if (S == 4) QH_SCE2(LM, 4); \
    else QH_SCE2(LM, 1);         \
  } while (0)
  switch (lMax) {
    case 1: QH_SCE(1); break;
    case 2: QH_SCE(2); break;
    case 3: QH_SCE(3); break;
    case 4: QH_SCE(4); break;
    default: qpms_hip_die(__FILE__, __LINE__, __func__, "lMax %d not instantiated (1..4)", lMax);
  }
#undef QH_SCE
#undef QH_SCE2
#undef QH_SCE1
  HIPCHK(hipGetLastError());
  return 0;
}
