// Point-wise physics shared by the HIP kernels: interpolation / well
// functions, face averages, the |grad q| floor, free energies and the per-cell
// KKS solve.  Operation order follows the reference Fortran so FP64 results
// agree with the CPU restatement to the last bits (transcendentals aside).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "../../include/ampe_hip.h"

#define AMPE_HD __host__ __device__ __forceinline__

#include "mathfn.h"

namespace ampe {

constexpr double kRGas = 8.314472;  // J/(K mol)

AMPE_HD double dmax(double a, double b) { return a > b ? a : b; }
AMPE_HD double dmin(double a, double b) { return a < b ? a : b; }

// interp_func (source/fortran/functions.f:17-92)
AMPE_HD double interp(double phi, char type)
{
   double t;
   switch (type) {
      case 'q': t = dmax(0.0, phi); return t * t;
      case 'p':
         t = dmax(0.0, dmin(1.0, phi));
         return t * t * t * (10.0 - 15.0 * t + 6.0 * t * t);
      case 'h':
         t = dmax(0.0, dmin(1.0, phi));
         return t * t * (3.0 - 2.0 * t);
      case 'w': t = dmax(0.0, phi); return t * t * (2.0 - t);
      case 'l':
         t = dmax(0.0, phi);
         t = dmin(1.0, t);
         return t;
      case 'm':
         t = dmax(0.0, dmin(1.0, phi));
         return t * t / (2.0 * t * (t - 1.0) + 1.0);
      case '3': t = dmax(0.0, phi); return t * t * t;
      case 's': return log(cosh(10.0 * phi)) / log(cosh(10.0));
      case 'c': return 1.0;
      default: return __builtin_nan("");
   }
}

// deriv_interp_func (source/fortran/functions.f:95-173)
AMPE_HD double dinterp(double phi, char type)
{
   double t, s;
   switch (type) {
      case 'q': t = dmax(0.0, phi); return 2.0 * t;
      case 'p':
         t = dmax(0.0, dmin(1.0, phi));
         return 30.0 * t * t * (1.0 - t) * (1.0 - t);
      case 'h':
         t = dmax(0.0, dmin(1.0, phi));
         return 6.0 * t * (1.0 - t);
      case 'w': t = dmax(0.0, phi); return t * (4.0 - 3.0 * t);
      // the reference tests phi > 0 .or. phi < 1 (functions.f:136-137), true for all phi
      case 'l': return (phi > 0.0 || phi < 1.0) ? 1.0 : 0.0;
      case 'm':
         t = dmax(0.0, dmin(1.0, phi));
         s = 2.0 * t * (t - 1.0) + 1.0;
         return 2.0 * t * (1.0 - t) / (s * s);
      case '3': t = dmax(0.0, phi); return 3.0 * t * t;
      case 's':
         t = dmax(0.0, phi);
         return 10.0 * tanh(10.0 * t) / log(cosh(10.0));
      case 'c': return 0.0;
      default: return __builtin_nan("");
   }
}

// deriv_well_func / second_deriv_well_func (source/fortran/functions.f:246-330)
AMPE_HD double dwell(double phi, char type)
{
   if (type == 'd') return 32.0 * phi * (1.0 - phi) * (1.0 - 2.0 * phi);
   return 2.0 * (phi - 1.0);
}
AMPE_HD double d2well(double phi, char type)
{
   if (type == 'd') return 32.0 * (1.0 + 6.0 * phi * (phi - 1.0));
   return 2.0;
}

// average_func (source/fortran/functions.f:333-365)
AMPE_HD double face_avg(double a, double b, char type)
{
   if (type == 'h') {
      if (a < 1.0e-16 || b < 1.0e-16) return 0.0;
      return 2.0 / (1.0 / a + 1.0 / b);
   }
   return 0.5 * (a + b);
}

// eval_grad_normi (source/fortran/quat.f:1497-1537).  x**(-0.5) is evaluated
// as 1/sqrt(x) (correctly rounded sqrt and divide: within 2 ulp of the power)
// instead of a general pow, which costs a log and an exp per face.
AMPE_HD double grad_normi(double gn2, char floor_type, double floor2,
                          double max_gni)
{
   if (floor_type == 'm') return (gn2 > floor2) ? 1.0 / sqrt(gn2) : max_gni;
   if (floor_type == 't') {
      double gng2 = gn2 * max_gni * max_gni;
      if (gng2 > 0.01) {
         double gn = sqrt(gn2);
         return tanh(max_gni * gn) / gn;
      }
      return max_gni * (1.0 - gng2 * (5.0 - 2.0 * gng2) / 15.0);
   }
   return 1.0 / sqrt(gn2 + floor2);
}

// quatmobility (source/fortran/2d/mobility.m4:13-90)
AMPE_HD double quat_mobility(const ampe_model_params& p, double ph)
{
   double qf;
   if (p.quat_mobility_type == 'e') {
      double c = p.quat_mobility_scale;
      ph = dmax(0.0, dmin(1.0, ph));
      qf = (1.0 - exp(c * ph)) / (1.0 - exp(c));
      qf = 1.0 - qf;
   } else if (p.quat_mobility_type == 'i') {
      ph = dmax(1.0e-6, dmin(1.0, ph));
      qf = dmax(0.0, (1.0 - ph) / (ph * ph));
      qf = dmin(qf, p.quat_mobility_scale);
   } else {
      ph = dmax(0.0, dmin(1.0, ph));
      qf = ph * ph * ph * (10.0 - 15.0 * ph + 6.0 * ph * ph);
      qf = 1.0 - qf;
   }
   return p.min_quat_mobility + (p.quat_mobility - p.min_quat_mobility) * qf;
}

// ---------------------------------------------------------------- energies
// Quadratic wells A (c - ceq(T))^2 and binary CALPHAD (end members, ideal
// mixing, Redlich-Kister excess), J/mol.  phase 0 = liquid, 1 = solid A.
AMPE_HD double quad_ceq(const ampe_model_params& p, int ph)
{
   return p.quad_ceq[ph] + p.quad_m[ph] * (p.temperature - p.quad_Tref);
}

// Binary CALPHAD phase at temperature T: G, dG/dc and d2G/dc2 [J/mol].
AMPE_HD double calphad_g(const ampe_calphad_phase& cp, double T, double c)
{
   double RT = kRGas * T;
   double x = 2.0 * c - 1.0;
   double P = cp.L[0] + x * (cp.L[1] + x * (cp.L[2] + x * cp.L[3]));
   return c * cp.gA + (1.0 - c) * cp.gB +
          RT * (c * log_pos(c) + (1.0 - c) * log_pos(1.0 - c)) + c * (1.0 - c) * P;
}

AMPE_HD double calphad_mu(const ampe_calphad_phase& cp, double T, double c)
{
   double RT = kRGas * T;
   double x = 2.0 * c - 1.0;
   double P = cp.L[0] + x * (cp.L[1] + x * (cp.L[2] + x * cp.L[3]));
   double dP = cp.L[1] + x * (2.0 * cp.L[2] + x * 3.0 * cp.L[3]);
   return cp.gA - cp.gB + RT * log_pos(c / (1.0 - c)) + (1.0 - 2.0 * c) * P +
          2.0 * c * (1.0 - c) * dP;
}

AMPE_HD double calphad_d2(const ampe_calphad_phase& cp, double T, double c)
{
   double RT = kRGas * T;
   double x = 2.0 * c - 1.0;
   double P = cp.L[0] + x * (cp.L[1] + x * (cp.L[2] + x * cp.L[3]));
   double dP = cp.L[1] + x * (2.0 * cp.L[2] + x * 3.0 * cp.L[3]);
   double d2P = 2.0 * cp.L[2] + x * 6.0 * cp.L[3];
   return RT / (c * (1.0 - c)) - 2.0 * P + 4.0 * (1.0 - 2.0 * c) * dP +
          4.0 * c * (1.0 - c) * d2P;
}

// Driving force (f_L(cl) - f_S(cs)) - mu_S(cs) (cl - cs) [J/mol] of the two
// CALPHAD phases.  With w(c) = f - c f' = G_B + RT ln(1 - c) + excess it is
// w_L(cl) - w_S(cs) + (mu_L(cl) - mu_S(cs)) cl: the logarithms pair up into two
// of quotients, where the energies and the potential one by one take five and
// cancel most of their digits against each other.
AMPE_HD double calphad_drive(const ampe_calphad_phase* ph, double T, double cl, double cs)
{
   const double RT = kRGas * T;
   const double l0 = log_ratio(1.0 - cl, 1.0 - cs), l1 = log_ratio(cl, cs);
   double w[2], mu[2];
   for (int k = 0; k < 2; k++) {
      const ampe_calphad_phase& q = ph[k];
      const double c = k == 0 ? cl : cs;
      const double x = 2.0 * c - 1.0;
      const double P = q.L[0] + x * (q.L[1] + x * (q.L[2] + x * q.L[3]));
      const double dP = q.L[1] + x * (2.0 * q.L[2] + x * 3.0 * q.L[3]);
      const double e = 2.0 * c * (1.0 - c) * dP - x * P;
      mu[k] = (q.gA - q.gB) + e;
      w[k] = q.gB + (c * (1.0 - c) * P - c * e);
   }
   return (w[0] - w[1]) + RT * l0 + ((mu[0] - mu[1]) + RT * (l1 - l0)) * cl;
}

// Dilute binary solution (c = solute fraction):
//   f_L(c) = RT (c ln c - c),
//   f_S(c) = RT (c ln c - c) - RT ln(k_e) c + dG(T),
//   dG(T)  = RT (k_e - 1)(T - T_m) / m,
// so mu_L = mu_S gives c_S = k_e c_L and the two-phase equilibrium lies on
// the linear liquidus c_L = (T - T_m) / m.
AMPE_HD double dilute_dG(const ampe_model_params& p)
{
   double RT = kRGas * p.temperature;
   return RT * (p.dilute_keq - 1.0) * (p.temperature - p.dilute_Tm) / p.dilute_m;
}

// Temperature-dependent parts of the CALPHAD atomic mobilities, per phase
// (0 liquid, 1 solid A) and species: Q_A, Q_B and the Redlich-Kister QQ_n of
// CALPHADMobility::getQ / getQQn (source/CALPHADMobility.h:42-103), formed on
// the host once per launch.
struct MobConst {
   double RT;
   double QA[2][2], QB[2][2];
   double QQ[2][2][4];
};

inline MobConst mob_const(const ampe_model_params& p)
{
   MobConst m;
   const double T = p.temperature;
   m.RT = kRGas * T;
   for (int ph = 0; ph < 2; ph++)
      for (int sp = 0; sp < 2; sp++) {
         const ampe_calphad_mobility& mb = p.mobility[ph][sp];
         double q[2];
         for (int x = 0; x < 2; x++) {
            q[x] = mb.q[x][0] + m.RT * std::log(mb.q[x][1]);
            if (mb.has_extra) q[x] += mb.qx[x][0] * T * std::log(T) + mb.qx[x][1] / T;
         }
         m.QA[ph][sp] = q[0];
         m.QB[ph][sp] = q[1];
         for (int n = 0; n < 4; n++)
            m.QQ[ph][sp][n] = mb.qq[n][0] + m.RT * std::log(mb.qq[n][1]);
      }
   return m;
}

// CALPHADMobility::getAtomicMobility for a binary (getDeltaG,
// source/CALPHADMobility.cc:155-166): exp(dG / RT) / RT.
AMPE_HD double atomic_mobility(const MobConst& m, int ph, int sp, double c0, double c1)
{
   const double dc = c0 - c1;
   const double* qq = m.QQ[ph][sp];
   const double dG = c0 * m.QA[ph][sp] + c1 * m.QB[ph][sp] +
                     c0 * c1 * (qq[0] + dc * (qq[1] + dc * (qq[2] + dc * qq[3])));
   const double rtinv = 1.0 / m.RT;
   return exp(dG * rtinv) * rtinv;
}

// computeDiffusionMobilityBinaryPhase (source/CALPHADMobility.cc:200-218):
// c0 c1 (c0 m1 + c1 m0), in um^2 (the 1e12 of m^2).
AMPE_HD double phase_diffusion_mobility(const MobConst& m, int ph, double c0)
{
   const double c1 = 1.0 - c0;
   const double m0 = atomic_mobility(m, ph, 0, c0, c1);
   const double m1 = atomic_mobility(m, ph, 1, c0, c1);
   const double mm = c0 * m1 + c1 * m0;
   return c0 * c1 * mm * 1.0e12;
}

// The energy functions take the model as a template argument FE when a kernel
// is specialised for it; FE < 0 reads p.fe_model at run time.
template <int FE>
AMPE_HD double fenergy_t(const ampe_model_params& p, double c, int ph)
{
   const int fe = (FE < 0) ? p.fe_model : FE;
   if (fe == AMPE_FE_QUADRATIC) {
      double d = c - quad_ceq(p, ph);
      return p.quad_A[ph] * d * d;
   }
   if (fe == AMPE_FE_KKS_DILUTE) {
      double RT = kRGas * p.temperature;
      double f = RT * (c * log_pos(c) - c);
      if (ph == 1) f = f - RT * log_pos(p.dilute_keq) * c + dilute_dG(p);
      return f;
   }
   return calphad_g(p.calphad[ph], p.temperature, c);
}

template <int FE>
AMPE_HD double dfenergy_t(const ampe_model_params& p, double c, int ph)
{
   const int fe = (FE < 0) ? p.fe_model : FE;
   if (fe == AMPE_FE_QUADRATIC) return 2.0 * p.quad_A[ph] * (c - quad_ceq(p, ph));
   if (fe == AMPE_FE_KKS_DILUTE) {
      double RT = kRGas * p.temperature;
      double mu = RT * log_pos(c);
      if (ph == 1) mu = mu - RT * log_pos(p.dilute_keq);
      return mu;
   }
   return calphad_mu(p.calphad[ph], p.temperature, c);
}

template <int FE>
AMPE_HD double d2fenergy_t(const ampe_model_params& p, double c, int ph)
{
   const int fe = (FE < 0) ? p.fe_model : FE;
   if (fe == AMPE_FE_QUADRATIC) return 2.0 * p.quad_A[ph];
   if (fe == AMPE_FE_KKS_DILUTE) return kRGas * p.temperature / c;
   return calphad_d2(p.calphad[ph], p.temperature, c);
}

AMPE_HD double fenergy(const ampe_model_params& p, double c, int ph)
{
   return fenergy_t<-1>(p, c, ph);
}
AMPE_HD double dfenergy(const ampe_model_params& p, double c, int ph)
{
   return dfenergy_t<-1>(p, c, ph);
}
AMPE_HD double d2fenergy(const ampe_model_params& p, double c, int ph)
{
   return d2fenergy_t<-1>(p, c, ph);
}

// Phase mobility at one cell: the uniform M_phi, or Kim's KKS mobility
// (KimMobilityStrategyInfMob::evaluateMobility, source/
// KimMobilityStrategyInfMob.cc:54-83; FiniteMob, KimMobilityStrategyFiniteMob.h
// :29-38; FiniteMobAntiTrap, .cc:54-80) with kks_mobility_factor
// (source/KKStools.cc:13-30) and zeta = (cL - cS) f_L''(cL) (cL - cS) / D_L(T)
// converted by 1e-6 / v_m.
template <int FE>
AMPE_HD double phase_mobility_t(const ampe_model_params& p, double cl, double cs)
{
   if (p.phi_mobility_type != AMPE_PHI_MOB_KIM) return p.phi_mobility;
   double eps = p.epsilon_phi, w = p.phi_well_scale;
   double a2 = (p.energy_interp == 'p') ? 47. / 60. : 0.5;
   double factor = 16. * w / (3. * eps * eps * a2);
   double alpha = 0.0;
   bool finite = p.kim_interface_mobility > 0.0;
   if (finite) {
      double xi = eps / sqrt(16. * w);
      alpha = 3. * sqrt(2.) * xi / p.kim_interface_mobility;
      if (!p.kim_antitrapping) return 1. / alpha;
   }
   double T = p.temperature;
   double DL = p.D_liquid * exp(-p.Q0_liquid / (kRGas * T));
   double d2 = d2fenergy_t<FE>(p, cl, 0);
   double zeta = 0.;
   zeta += (cl - cs) * d2 * (cl - cs);
   double zf = zeta / DL;
   zf *= (1.e-6 / p.vm_L);
   if (finite) return 1. / (alpha + (1. / factor) * zf);
   return factor / zf;
}

AMPE_HD double phase_mobility(const ampe_model_params& p, double cl, double cs)
{
   return phase_mobility_t<-1>(p, cl, cs);
}

// End-member G(T) of a tdep table: interval k is the last with T >= Tc[k]
// (k <= nrange - 1); terms added in database order.
AMPE_HD double calphad_gfun(const ampe_calphad_gfun& f, double T)
{
   int k = 0;
   while (k < f.nrange - 1 && T >= f.Tc[k + 1]) k++;
   const double* a = f.coef[k];
   double T2 = T * T, T3 = T2 * T;
   double T7 = T3 * T3 * T;
   double Tm9 = 1.0 / (T3 * T3 * T3);
   double g = a[0] + a[1] * T + a[2] * T * log_pos(T);
   g = g + a[3] * T2;
   g = g + a[4] * T3;
   g = g + a[5] * T7;
   g = g + a[6] / T;
   g = g + a[7] * Tm9;
   return g;
}

AMPE_HD void calphad_at(const ampe_calphad_tdep& tab, double T, ampe_calphad_phase* out)
{
   for (int ph = 0; ph < 2; ph++) {
      out[ph].gA = calphad_gfun(tab.g[ph][0], T);
      out[ph].gB = calphad_gfun(tab.g[ph][1], T);
      for (int i = 0; i < 4; i++) out[ph].L[i] = tab.L[ph][i][0] + tab.L[ph][i][1] * T;
   }
}

// What the binary CALPHAD KKS system needs of the two phases at one
// temperature, over RT: the difference of the end members' G_A - G_B, and the
// excess part of dG/dc as a polynomial in u = 2c - 1 (with P the Redlich-Kister
// sum, (1 - 2c) P + 2c(1 - c) P' = -u P + (1 - u^2)/2 P').
struct KksTerms {
   double k0;
   double e[2][5];
};

AMPE_HD void kks_excess(const double* L, double RTinv, double* e)
{
   e[0] = 0.5 * L[1] * RTinv;
   e[1] = (L[2] - L[0]) * RTinv;
   e[2] = 1.5 * (L[3] - L[1]) * RTinv;
   e[3] = -2.0 * L[2] * RTinv;
   e[4] = -2.5 * L[3] * RTinv;
}

AMPE_HD KksTerms kks_terms(const ampe_calphad_phase* ph, double T)
{
   const double RTinv = 1.0 / (kRGas * T);
   KksTerms t;
   t.k0 = ((ph[0].gA - ph[0].gB) - (ph[1].gA - ph[1].gB)) * RTinv;
   for (int k = 0; k < 2; k++) kks_excess(ph[k].L, RTinv, t.e[k]);
   return t;
}

// Residual of the binary CALPHAD KKS system at (xl, xs):
// F = [(mu_L(xl) - mu_S(xs))/RT, (1-h) xl + h xs - c].  The two ideal parts
// are one logarithm, ln(xl (1 - xs) / ((1 - xl) xs)).
AMPE_HD void kks_residual(const KksTerms& t, double h, double c, double xl, double xs, double& f1,
                          double& f2)
{
   const double u = std::fma(2.0, xl, -1.0), v = std::fma(2.0, xs, -1.0);
   const double* a = t.e[0];
   const double* b = t.e[1];
   const double el =
       std::fma(u, std::fma(u, std::fma(u, std::fma(u, a[4], a[3]), a[2]), a[1]), a[0]);
   const double es =
       std::fma(v, std::fma(v, std::fma(v, std::fma(v, b[4], b[3]), b[2]), b[1]), b[0]);
   f1 = (t.k0 + (el - es)) + log_ratio(xl * (1.0 - xs), (1.0 - xl) * xs);
   f2 = (1.0 - h) * xl + h * xs - c;
}

// The terms at a cell's temperature from a tdep table, the end members by
// calphad_gfun's intervals and terms.  The interval loop is uniform and a
// lane enters the intervals its temperature lies in (one or two over a wave), so
// that the coefficients are scalars; indexing them by the lane's interval
// costs 32 gathered loads a cell.  (The terms are summed as calphad_gfun sums
// them: those of one end member reach 10^6 J/mol and cancel, and another order
// moves the potentials by 1e-14 RT.)
AMPE_HD KksTerms kks_terms_at(const ampe_calphad_tdep& tab, double T)
{
   const double Ti = 1.0 / T, lnT = log_pos(T);
   const double T2 = T * T, T3 = T2 * T, T7 = T3 * T3 * T;
   const double Tm9 = 1.0 / (T3 * T3 * T3);
   double g[2][2];
   for (int ph = 0; ph < 2; ph++)
      for (int sp = 0; sp < 2; sp++) {
         const ampe_calphad_gfun& f = tab.g[ph][sp];
         bool above = true;  // T >= Tc[1..k]
         double v = 0.0;
         for (int k = 0; k < f.nrange; k++) {
            const bool next = k < f.nrange - 1 && T >= f.Tc[k + 1];
            if (above && !next) {
               const double* a = f.coef[k];
               v = a[0] + a[1] * T + a[2] * T * lnT;
               v = v + a[3] * T2;
               v = v + a[4] * T3;
               v = v + a[5] * T7;
               v = v + a[6] * Ti;
               v = v + a[7] * Tm9;
            }
            above = above && next;
         }
         g[ph][sp] = v;
      }
   const double RTinv = 1.0 / (kRGas * T);
   KksTerms t;
   t.k0 = ((g[0][0] - g[0][1]) - (g[1][0] - g[1][1])) * RTinv;
   for (int ph = 0; ph < 2; ph++) {
      double L[4];
      for (int i = 0; i < 4; i++) L[i] = std::fma(tab.L[ph][i][1], T, tab.L[ph][i][0]);
      kks_excess(L, RTinv, t.e[ph]);
   }
   return t;
}

// Start of a KKS Newton: the guess clamped into [1e-12, 1-1e-12].
AMPE_HD void kks_clamp(double& xl, double& xs)
{
   const double lo = 1.0e-12, hi = 1.0 - 1.0e-12;
   if (!(xl > lo)) xl = lo;
   if (!(xl < hi)) xl = hi;
   if (!(xs > lo)) xs = lo;
   if (!(xs < hi)) xs = hi;
}

// Newton iterations from a clamped start (xl, xs) whose residual (f1, f2) is
// given; step halving keeps the iterate inside (0,1); converged when both
// |F_i| < tol.  Returns the number of updates, -1 after maxits updates
// without convergence, or -2 when probe_its >= 0 and max|F| > probe_tol after
// probe_its updates (the caller restarts).  The test stops a hundredth short of
// tol: the residual's rounding (about 1e-15 of the ideal and excess parts)
// depends on the order of its terms, and a solution accepted here is within tol
// in any order.
// The solve is bound by FP64 arithmetic: an update is one logarithm and two
// divisions (the Jacobian 1/(x (1 - x)) + E'(x) of each phase enters multiplied by
// both x (1 - x)), against two logarithms of quotients and eight divisions with
// each phase's potential and second derivative evaluated by itself.
AMPE_HD int kks_newton_from(const KksTerms& t, double h, double c, double& cl, double& cs,
                            double f1, double f2, int maxits, double tol, int probe_its,
                            double probe_tol)
{
   double xl = cl, xs = cs;
   const double accept = 0.99 * tol;
   for (int it = 0; it <= maxits; it++) {
      if (it > 0) kks_residual(t, h, c, xl, xs, f1, f2);
      if (fabs(f1) < accept && fabs(f2) < accept) {
         cl = xl;
         cs = xs;
         return it;
      }
      if (it == maxits) break;
      if (it == probe_its && !(dmax(fabs(f1), fabs(f2)) <= probe_tol)) {
         cl = xl;
         cs = xs;
         return -2;
      }
      const double u = std::fma(2.0, xl, -1.0), v = std::fma(2.0, xs, -1.0);
      const double* a = t.e[0];
      const double* b = t.e[1];
      // dE/dc = 2 dE/du
      const double dl2 =
          std::fma(u, std::fma(u, std::fma(u, 8.0 * a[4], 6.0 * a[3]), 4.0 * a[2]), 2.0 * a[1]);
      const double ds2 =
          std::fma(v, std::fma(v, std::fma(v, 8.0 * b[4], 6.0 * b[3]), 4.0 * b[2]), 2.0 * b[1]);
      const double pl = xl * (1.0 - xl), ps = xs * (1.0 - xs);
      const double A = ps * std::fma(pl, dl2, 1.0), S = pl * std::fma(ps, ds2, 1.0);
      const double q1 = pl * ps * f1;
      const double inv = 1.0 / std::fma(A, h, S * (1.0 - h));
      const double dl = -std::fma(h, q1, S * f2) * inv;
      const double ds = -std::fma(A, f2, -(1.0 - h) * q1) * inv;
      double alpha = 1.0;
      for (int k = 0; k < 60; k++) {
         double nl = xl + alpha * dl, ns = xs + alpha * ds;
         if (nl > 0.0 && nl < 1.0 && ns > 0.0 && ns < 1.0) break;
         alpha *= 0.5;
      }
      xl = xl + alpha * dl;
      xs = xs + alpha * ds;
   }
   cl = xl;
   cs = xs;
   return -1;
}

// Binary CALPHAD KKS Newton from the guess (cl, cs) (see kks_newton_from).
AMPE_HD int kks_newton(const KksTerms& t, double h, double c, double& cl, double& cs, int maxits,
                       double tol, int probe_its, double probe_tol)
{
   kks_clamp(cl, cs);
   double f1, f2;
   kks_residual(t, h, c, cl, cs, f1, f2);
   return kks_newton_from(t, h, c, cl, cs, f1, f2, maxits, tol, probe_its, probe_tol);
}

// Quadratic wells: closed form of mu_L = mu_S with mass balance.
AMPE_HD void kks_quadratic(const ampe_model_params& p, double h, double c, double& cl,
                           double& cs)
{
   double eL = quad_ceq(p, 0), eS = quad_ceq(p, 1);
   double r = p.quad_A[0] / p.quad_A[1];
   double xl = (c - h * (eS - r * eL)) / (1.0 - h + h * r);
   cl = xl;
   cs = eS + r * (xl - eL);
}

// Per-cell KKS at the model temperature: mu_L(cL) = mu_S(cS),
// (1-h) cL + h cS = c.  Quadratic wells and the dilute solution: closed
// forms.  CALPHAD: kks_newton from the guess in (cl, cs) with the phases' terms
// t.  Returns the iteration count or -1.
template <int FE>
AMPE_HD int kks_cell(const ampe_model_params& p, const KksTerms& t, double c, double phi,
                     double& cl, double& cs)
{
   double h = interp(phi, p.conc_interp);
   if (FE == AMPE_FE_QUADRATIC) {
      kks_quadratic(p, h, c, cl, cs);
      return 0;
   }
   if (FE == AMPE_FE_KKS_DILUTE) {
      double k = p.dilute_keq;
      double xl = c / (1.0 - h + h * k);
      cl = xl;
      cs = k * xl;
      return 0;
   }
   return kks_newton(t, h, c, cl, cs, p.newton_max_its, p.newton_tol, -1, 0.0);
}

}  // namespace ampe
