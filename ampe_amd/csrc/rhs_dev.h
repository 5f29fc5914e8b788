// Face and cell terms shared by the right-hand-side kernels.
#pragma once

#include "kernels.h"

namespace ampe {

// Single precision literal 1.e-12 of anisotropic_gradient_flux promoted to
// double (source/fortran/2d/quatrhs.m4:193, 3d/quatrhs.m4:184).
#define AMPE_ANISO_THRESHOLD ((double)1.e-12f)

// ------------------------------------------------------------ phase flux
// Face between cells cm = c0 - st[d] and c0, direction d.
// Simple: gradient_flux (source/fortran/2d/quatrhs.m4:12-53).
// Isotropic (2-D): compute_flux_isotropic (2d/quatrhs.m4:106-151).
// Anisotropic: anisotropic_gradient_flux (2d/quatrhs.m4:154-256,
// 3d/quatrhs.m4:149-356).
__device__ __forceinline__ void quatmult4(const double* a, const double* b, double* r)
{
   r[0] = a[0] * b[0] - a[1] * b[1] - a[2] * b[2] - a[3] * b[3];
   r[1] = a[0] * b[1] + a[1] * b[0] + a[2] * b[3] - a[3] * b[2];
   r[2] = a[0] * b[2] + a[2] * b[0] + a[3] * b[1] - a[1] * b[3];
   r[3] = a[0] * b[3] + a[3] * b[0] + a[1] * b[2] - a[2] * b[1];
}

// cos and sin of kn (theta - phi): theta = atan(gy / gx) in (-pi/2, pi/2), pi/2 for
// |gx| at or below the threshold; phi = acos(qa), twice that with `twice`.  The unit
// vectors of theta and phi are algebraic in the arguments, their quotient's kn-th
// power has the cosine and sine wanted: two square roots, a division and some
// products for the four transcendentals (atan, acos, cos, sin) of the angle form.
// 1 - qa^2 is formed as (1 - qa)(1 + qa), exact to rounding near the ends, where
// acos is steep; the error of the cosine and sine against extended
// precision is 1.1e-15 at most for kn = 4 and 1.7e-15 for 6 (angle form 3.9e-15 and
// 9.1e-15), 0.2e-15 and 0.3e-15 in the mean square (0.5e-15 and 0.9e-15), over
// 4 10^5 directions and angles, half of them with qa near 1.
// 1500 x 1130 dendrite, full right-hand side: 81 us (98 in the angle form with
// the logarithm of k_e taken in every cell).
__device__ __forceinline__ void aniso_angle(double gx, double gy, double qa, bool twice, int kn,
                                            double& cs, double& sn)
{
   double ct = 0.0, st = 1.0;
   if (fabs(gx) > AMPE_ANISO_THRESHOLD) {
      const double ri = 1.0 / sqrt(gx * gx + gy * gy);
      ct = fabs(gx) * ri;
      st = (gx < 0.0 ? -gy : gy) * ri;
   }
   double cp = qa, sp = sqrt((1.0 - qa) * (1.0 + qa));
   if (twice) {
      sp = 2.0 * qa * sp;
      cp = fma(2.0 * qa, qa, -1.0);
   }
   // exp(i (theta - phi)), its modulus put back to one: rounding moved it by an
   // ulp or two, and the power would by kn times that
   double x = ct * cp + st * sp, y = st * cp - ct * sp;
   const double e = -0.5 * fma(x, x, fma(y, y, -1.0));
   x = fma(e, x, x);
   y = fma(e, y, y);
   const int n = kn < 0 ? -kn : kn;
   cs = 1.0;
   sn = 0.0;
   for (int m = n; m > 0; m >>= 1) {
      if (m & 1) {
         const double u = fma(cs, x, -(sn * y));
         sn = fma(cs, y, sn * x);
         cs = u;
      }
      const double v = fma(x, x, -(y * y));
      y = 2.0 * x * y;
      x = v;
   }
   if (kn < 0) sn = -sn;
}

// FLUX < 0 reads p.flux_type at run time.
template <int NDIM, int FLUX = -1>
__device__ double phase_face_flux(const ampe_model_params& p, const RhsConst& k,
                                  const double* __restrict__ ph, const double* __restrict__ q,
                                  long long ncg, const long long* st, int d, long long cm,
                                  long long c0)
{
   const int ft = (FLUX < 0) ? p.flux_type : FLUX;
   if (ft == AMPE_FLUX_ANISOTROPIC) {
      if (NDIM == 2) {
         double eps = p.epsilon_phi, nu = p.aniso_nu;
         int kn = p.aniso_knumber;
         double dinv0 = k.dxinv[0], dinv1 = k.dxinv[1];
         int t = 1 - d;  // transverse direction
         double gn = (ph[c0] - ph[cm]) * (d == 0 ? dinv0 : dinv1);
         double gt = 0.25 * (ph[cm + st[t]] - ph[cm - st[t]] + ph[c0 + st[t]] - ph[c0 - st[t]]) *
                     (d == 0 ? dinv1 : dinv0);
         double dphidx = (d == 0) ? gn : gt;
         double dphidy = (d == 0) ? gt : gn;
         double qa = 0.5 * (q[cm] + q[c0]);
         if (qa > 1.0) qa = 1.0;
         if (qa < -1.0) qa = -1.0;
         double cs, sn;
         aniso_angle(dphidx, dphidy, qa, p.qlen == 4, kn, cs, sn);
         double epst = eps * (1.0 + nu * cs);
         double deps = -kn * eps * nu * sn;
         if (d == 0) return epst * epst * dphidx - epst * deps * dphidy;
         return epst * epst * dphidy + epst * deps * dphidx;
      } else {
         double eps = p.epsilon_phi, eps4 = p.aniso_nu;
         const double* dinv = k.dxinv;
         double factor = 4.0 * eps4 / (1.0 - 3.0 * eps4);
         double gr[3];
#pragma unroll
         for (int e = 0; e < 3; e++) {
            if (e == d)
               gr[e] = (ph[c0] - ph[cm]) * dinv[e];
            else
               gr[e] = 0.25 * (ph[cm + st[e]] - ph[cm - st[e]] + ph[c0 + st[e]] - ph[c0 - st[e]]) *
                       dinv[e];
         }
         double gphi2 = gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2];
         double dg[4], n4;
         if (fabs(gphi2) > AMPE_ANISO_THRESHOLD) {
            double nni = 1.0 / sqrt(gphi2);
            double n[4] = {0.0, gr[0] * nni, gr[1] * nni, gr[2] * nni};
            double qa[4];
#pragma unroll
            for (int m = 0; m < 4; m++) qa[m] = 0.5 * (q[m * ncg + cm] + q[m * ncg + c0]);
            double qp[4] = {qa[0], -qa[1], -qa[2], -qa[3]}, tq[4], np[4];
            quatmult4(n, qp, tq);
            quatmult4(qa, tq, np);
            double a1 = np[1] * np[1], a2 = np[2] * np[2], a3 = np[3] * np[3];
            n4 = a1 * a1 + a2 * a2 + a3 * a3;
            double dd[4] = {0.0, np[1] * (np[1] * np[1] - n4), np[2] * (np[2] * np[2] - n4),
                            np[3] * (np[3] * np[3] - n4)};
            quatmult4(dd, qa, tq);
            quatmult4(qp, tq, dg);
         } else {
            dg[0] = dg[1] = dg[2] = dg[3] = 0.0;
            n4 = 0.0;
         }
         double gamma = eps * (1.0 - 3.0 * eps4) * (1.0 + factor * n4);
         return gamma * gamma * gr[d] + 16.0 * eps * gamma * eps4 * sqrt(gphi2) * dg[d + 1];
      }
   }
   if (ft == AMPE_FLUX_ISOTROPIC && NDIM == 2) {
      double dinv = k.e2dx12[d];
      long long t = st[1 - d];
      return dinv * ((ph[c0 - t] - ph[cm - t]) + (ph[c0] - ph[cm]) * 10.0 + (ph[c0 + t] - ph[cm + t]));
   }
   return (ph[c0] - ph[cm]) * k.e2dx[d];
}

// |grad q|^2 on faces from the full side gradient (quatgrad_side
// 2d/quatgrad.m4:157-229, summed as compute_face_coef2d quatfacops.m4:83-92).
template <int NDIM>
__device__ __forceinline__ double quat_face_norm2(const ampe_model_params& p, const RhsConst& k,
                                                  const double* __restrict__ q, long long ncg,
                                                  const long long* st, int d, long long cm,
                                                  long long c0)
{
   double s = 0.0;
   const int ql = p.qlen;
#pragma unroll
   for (int n = 0; n < NDIM; n++) {
      double dinv = k.dxinv[n];
      double p25 = 0.25 * dinv;
#pragma unroll
      for (int m = 0; m < ql; m++) {
         const double* aa = q + m * ncg;
         double gv;
         if (n == d) {
            gv = dinv * (aa[c0] - aa[cm]);
         } else {
            long long t = st[n];
            gv = p25 * ((aa[cm + t] - aa[cm]) + (aa[cm] - aa[cm - t]) + (aa[c0 + t] - aa[c0]) +
                        (aa[c0] - aa[c0 - t]));
         }
         s = s + gv * gv;
      }
   }
   return s;
}

// interp, dinterp and face_avg of N arguments with one test of the type: the
// type is the same for the whole launch, but a branch per evaluation (some
// thirty a cell in the fused kernel) kept loads and arithmetic of different
// faces apart.
template <int N>
__device__ __forceinline__ void interp_n(const double (&x)[N], double (&r)[N], char type)
{
   auto all = [&](char t) {
#pragma unroll
      for (int i = 0; i < N; i++) {
         r[i] = interp(x[i], t);
         // one transcendental after the other: together they would take the
         // registers of the whole kernel
         if (t == 's' || t == 'm') __builtin_amdgcn_sched_barrier(0);
      }
   };
   switch (type) {
      case 'q': return all('q');
      case 'p': return all('p');
      case 'h': return all('h');
      case 'l': return all('l');
      case 'c': return all('c');
      case 'w': return all('w');
      case '3': return all('3');
      case 'm': return all('m');
      case 's': return all('s');
      default: return all(0);
   }
}

template <int N>
__device__ __forceinline__ void dinterp_n(const double (&x)[N], double (&r)[N], char type)
{
   auto all = [&](char t) {
#pragma unroll
      for (int i = 0; i < N; i++) {
         r[i] = dinterp(x[i], t);
         // one transcendental after the other: together they would take the
         // registers of the whole kernel
         if (t == 's' || t == 'm') __builtin_amdgcn_sched_barrier(0);
      }
   };
   switch (type) {
      case 'q': return all('q');
      case 'p': return all('p');
      case 'h': return all('h');
      case 'l': return all('l');
      case 'c': return all('c');
      case 'w': return all('w');
      case '3': return all('3');
      case 'm': return all('m');
      case 's': return all('s');
      default: return all(0);
   }
}

template <int N>
__device__ __forceinline__ void face_avg_n(const double (&x)[N], double y, double (&r)[N],
                                           char type)
{
   auto all = [&](char t) {
#pragma unroll
      for (int i = 0; i < N; i++) r[i] = face_avg(x[i], y, t);
   };
   if (type == 'h')
      all('h');
   else
      all('a');
}

// compute_face_coef2d/3d (2d/quatfacops.m4:14-122) from the face |grad q|^2's
// 1 / |grad q| (grad_normi), and from |grad q|^2 itself.
__device__ __forceinline__ double quat_face_coef_gni(const ampe_model_params& p, double phm,
                                                     double ph0, double gni)
{
   double eps2 = p.epsilon_q * p.epsilon_q;
   double mf = 2.0 * p.H_parameter;
   double phia = face_avg(phm, ph0, p.avg_type);
   double tempa = 0.5 * (p.temperature + p.temperature);
   double diff = mf * tempa * interp(phia, p.orient_interp1);
   double hphi2 = interp(phia, p.orient_interp2);
   return -gni * diff - eps2 * hphi2;
}

__device__ __forceinline__ double face_gni(const ampe_model_params& p, const RhsConst& k,
                                           double n2f)
{
   return grad_normi(n2f, p.floor_type, p.gradient_floor * p.gradient_floor, k.maxgni);
}

__device__ __forceinline__ double quat_face_coef(const ampe_model_params& p, const RhsConst& k,
                                                 double phm, double ph0, double n2f)
{
   return quat_face_coef_gni(p, phm, ph0, face_gni(p, k, n2f));
}

// KKS driving force (QuadraticFreeEnergyStrategy.cc:393-511,
// CALPHADFreeEnergyStrategyBinary.cc:521-651).  kFeNone: no composition field.
constexpr int kFeNone = 3;

template <int FE>
__device__ __forceinline__ double phase_drive(const ampe_model_params& p, const RhsConst& k,
                                              double ph, double c_l, double c_a)
{
   const double convL = k.convL, convA = k.convA;
   const double hp = dinterp(ph, p.energy_interp);
   if (FE == AMPE_FE_CALPHAD_BINARY && convL == convA)
      return hp * (calphad_drive(p.calphad, p.temperature, c_l, c_a) * convL);
   if (FE == AMPE_FE_KKS_DILUTE) {
      // fenergy and dfenergy with the constants' logarithm and division on the host
      const double RT = kRGas * p.temperature, ls = log_pos(c_a);
      const double f_l = RT * (c_l * log_pos(c_l) - c_l) * convL;
      const double f_a = (RT * (c_a * ls - c_a) - RT * k.logk * c_a + k.dG) * convA;
      const double mu = (RT * ls - RT * k.logk) * convA;
      return hp * ((f_l - f_a) - mu * (c_l - c_a));
   }
   const double f_l = fenergy_t<FE>(p, c_l, 0) * convL;
   const double f_a = fenergy_t<FE>(p, c_a, 1) * convA;
   const double mu = (FE == AMPE_FE_QUADRATIC) ? dfenergy_t<FE>(p, c_l, 0) * convL
                                               : dfenergy_t<FE>(p, c_a, 1) * convA;
   return hp * ((f_l - f_a) - mu * (c_l - c_a));
}

// Dc and Dphi of the face between cells m and 0: concentration_pfmdiffusion
// (2d/concentrationdiffusion.m4:14-96) and setDiffCoeffForPhaseOnPatch
// (source/KKSCompositionRHSStrategy.cc:210-373).
__device__ __forceinline__ void conc_face_coeffs(const ampe_model_params& p, const RhsConst& k,
                                                 double phm, double ph0, double clm, double cl0,
                                                 double csm, double cs0, double& Dc, double& Dphi)
{
   const double ph = face_avg(phm, ph0, p.avg_type);
   const double hphi = interp(ph, p.energy_interp);
   const double dd = (1.0 - hphi) * k.Dl + hphi * k.Ds;
   const double c_l = 0.5 * (cl0 + clm);
   const double c_a = 0.5 * (cs0 + csm);
   Dc = dd;
   Dphi = dd * dinterp(ph, p.energy_interp) * (c_l - c_a);
}

}  // namespace ampe
