// The integrator's right-hand side of one level, or of all levels of a hierarchy
// at once, in one launch: phase (PhaseRHSStrategyWithQ::evaluateRHS), orientation
// (QuatFACOps::evaluateRHS with projection) and, in the KKS form, composition
// (KKSCompositionRHSStrategy).
//
// Each of the three reads phi's and two of them q's 7-point (5-point)
// neighbourhoods; one after the other they read both twice and passed the face
// coefficients of the orientation operator through memory (48 bytes a cell).
// Here a thread forms everything for its cell from one set of loads: the
// orientation's face coefficients take the face's 1 / |grad q|, which is lagged
// (it changes at full evaluations only), so that a coefficient is a few products
// and is cheaper formed from both sides than stored.  The operations and their
// order are those of the separate kernels (k_phase_rhs, k_quat_rhs, k_conc_rhs,
// k_conc_coeffs), and so are the values.
//
// 256^3, CALPHAD, full evaluation: 1116 us (184 bytes a cell, 2.8 TB/s); the five
// separate kernels took 1884 us.  Bound by latency at three wavefronts a SIMD
// (155 registers): a bound of 128 registers spills (1736 us), and a thread that
// goes on to the next planes holds back the loads behind its stores (2671 us for
// one plane a thread in that form).  Lagged on 151 x 93 x 67: 71 us.  Anisotropic
// dilute alloy, 1500 x 1130: 81 us (98 with a face angle from four transcendentals
// and the logarithm of k_e taken in every cell).
#include <type_traits>

#include "krylov.h"
#include "rhs_dev.h"

namespace ampe {

namespace {

// FIN: the right-hand side is a difference quotient's, and goes on to the
// preconditioner's input (KryFin) without being stored.  128^3, six components:
// 85 us less per Krylov iteration of 1.2 ms than storing it for a launch that reads
// it; 128^2: two launches fewer of nineteen with the ghosts filled by the kernel
// that forms the state.
template <int NDIM, int FE, int CONC, bool FIN>
__device__ __forceinline__ void rhs_tail(const LevelArgs& a, const ampe_model_params& p,
                                         const RhsConst& k, const CellPos& c, double r,
                                         const double* __restrict__ phi,
                                         const double* __restrict__ q,
                                         const double* __restrict__ cc,
                                         const double* __restrict__ cl,
                                         const double* __restrict__ cs,
                                         const double* __restrict__ gni, double* __restrict__ Dc,
                                         double* __restrict__ Dphi, double* __restrict__ yp,
                                         double* __restrict__ yq, double* __restrict__ yc,
                                         const KryFin& fin, int iq, int ic)
{
   const long long c0 = c.c0, ncg = a.ncg;
   long long sp = 0;
   double sm = 1.0;
   if (FIN) {
      if (fin.pin.sp0 < (1 << 30)) sp = split_at(a, c, 0);
      if (fin.pin.sm) sm = fin.pin.sm[c0];
   }
   // component m of the state vector, at field y's entry i
   auto put = [&](double* y, long long i, int m, double v) {
      if (FIN)
         prec_in(a, fin.pin, c, sp, m, kry_fin(fin, m * ncg + c0, v), sm, fin.out);
      else
         y[i] = v;
   };
   const double* dinv = k.dxinv;
   const double* hd = k.hdxinv;
   constexpr int NF = 2 * NDIM;  // faces: low of direction d at d, high at NDIM + d
   const double ph = phi[c0];
   double phn[NF];
   long long fi[NF], cn[NF];
   const int ijk[3] = {c.i, c.j, c.k};
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      int lo[3] = {ijk[0], ijk[1], ijk[2]};
      fi[d] = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      lo[d] += 1;
      fi[NDIM + d] = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      cn[d] = c0 - c.st[d];
      cn[NDIM + d] = c0 + c.st[d];
      phn[d] = phi[cn[d]];
      phn[NDIM + d] = phi[cn[NDIM + d]];
   }
   double pha[NF];
   face_avg_n(phn, ph, pha, p.avg_type);
   r = r - p.phi_well_scale * dwell(ph, p.phi_well_type);
   if (q) {
      // quat_face_coef_gni of the faces
      double fc[NF];
      {
         const double eps2 = p.epsilon_q * p.epsilon_q;
         const double mft = 2.0 * p.H_parameter * (0.5 * (p.temperature + p.temperature));
         double i1[NF], i2[NF];
         interp_n(pha, i1, p.orient_interp1);
         interp_n(pha, i2, p.orient_interp2);
#pragma unroll
         for (int e = 0; e < NF; e++) fc[e] = -gni[fi[e]] * (mft * i1[e]) - eps2 * i2[e];
      }
      double g2 = 0.0, lam = 0.0, sumq2 = 0.0, dv[4], qv[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
         const double* aa = q + m * ncg;
         const double qm = aa[c0];
         double gr[NDIM], dif[NDIM];
#pragma unroll
         for (int d = 0; d < NDIM; d++) {
            const double dl = qm - aa[cn[d]], dh = aa[cn[NDIM + d]] - qm;
            gr[d] = (dh + dl) * hd[d];
            dif[d] = fc[NDIM + d] * (dinv[d] * dh) - fc[d] * (dinv[d] * dl);
         }
         if (NDIM == 3) {
            g2 = g2 + gr[0] * gr[0] + gr[1] * gr[1] + gr[NDIM - 1] * gr[NDIM - 1];
            lam = lam - qm * (dif[0] * hd[0] + dif[1] * hd[1] + dif[NDIM - 1] * hd[NDIM - 1]);
            dv[m] = dif[0] * dinv[0] + dif[1] * dinv[1] + dif[NDIM - 1] * dinv[NDIM - 1];
         } else {
            g2 = g2 + gr[0] * gr[0] + gr[1] * gr[1];
            lam = lam - qm * (dif[0] * hd[0] + dif[1] * hd[1]);
            dv[m] = dif[0] * dinv[0] + dif[1] * dinv[1];
         }
         sumq2 = sumq2 + qm * qm;
         qv[m] = qm;
      }
      lam = lam / sumq2;
      const double mq = quat_mobility(p, ph);
#pragma unroll
      for (int m = 0; m < 4; m++)
         put(yq, m * ncg + c0, iq + m, 0.0 - mq * (dv[m] + 2.0 * qv[m] * lam));
      const double mf = 2.0 * p.H_parameter, T = p.temperature;
      const double eq2 = 0.5 * p.epsilon_q * p.epsilon_q;
      const double gm = sqrt(g2);
      r = r - mf * T * dinterp(ph, p.orient_interp1) * gm -
          dinterp(ph, p.orient_interp2) * eq2 * gm * gm;
   }
   double mob = p.phi_mobility;
   if (FE != kFeNone) {
      r += phase_drive<FE>(p, k, ph, cl[c0], cs[c0]);
      if (p.phi_mobility_type == AMPE_PHI_MOB_KIM) mob = phase_mobility_t<FE>(p, cl[c0], cs[c0]);
   }
   put(yp, c0, 0, mob * r);
   if (CONC == 0) return;
   const double cv = cc[c0];
   double Df[NF], Ef[NF];  // Dc and Dphi of the faces
   if (CONC == 1) {
#pragma unroll
      for (int e = 0; e < NF; e++) {
         Df[e] = Dc[fi[e]];
         Ef[e] = Dphi[fi[e]];
      }
   } else {
      // conc_face_coeffs of the faces
      double h[NF], hp[NF];
      interp_n(pha, h, p.energy_interp);
      dinterp_n(pha, hp, p.energy_interp);
      const double l0 = cl[c0], s0 = cs[c0];
      const int n[3] = {c.pd.nx, c.pd.ny, c.pd.nz};
#pragma unroll
      for (int e = 0; e < NF; e++) {
         Df[e] = (1.0 - h[e]) * k.Dl + h[e] * k.Ds;
         Ef[e] = Df[e] * hp[e] * (0.5 * (l0 + cl[cn[e]]) - 0.5 * (s0 + cs[cn[e]]));
         const int d = e % NDIM;
         if (e < NDIM || ijk[d] == n[d] - 1) {
            Dc[fi[e]] = Df[e];
            Dphi[fi[e]] = Ef[e];
         }
      }
   }
   double s = 0.0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      const double jl = dinv[d] * (Df[d] * (cv - cc[cn[d]]) + Ef[d] * (ph - phn[d]));
      const double jh = dinv[d] * (Df[NDIM + d] * (cc[cn[NDIM + d]] - cv) +
                                   Ef[NDIM + d] * (phn[NDIM + d] - ph));
      const double t = dinv[d] * (jh - jl);
      s = (d == 0) ? t : s + t;
   }
   put(yc, c0, ic, p.conc_mobility * s);
}

// One cell per thread; the anisotropic flux (square roots, a division and a
// power a face) is evaluated once per x and y face through LDS
// (k_phase_rhs_faces).
template <int NDIM, int FLUX, int FE, int CONC, bool FIN>
__global__ void __launch_bounds__(256) k_rhs_all(LevelArgs a, ampe_model_params p, RhsLev kl,
                                                 const double* __restrict__ phi,
                                                 const double* __restrict__ q,
                                                 const double* __restrict__ cc,
                                                 const double* __restrict__ cl,
                                                 const double* __restrict__ cs,
                                                 const double* __restrict__ gni,
                                                 double* __restrict__ Dc,
                                                 double* __restrict__ Dphi,
                                                 double* __restrict__ yp, double* __restrict__ yq,
                                                 double* __restrict__ yc, KryFin fin, int iq,
                                                 int ic)
{
   if constexpr (FLUX == AMPE_FLUX_ANISOTROPIC) {
      __shared__ double fx[TY][TX + 1];
      __shared__ double fy[TY + 1][TX];
      const Tile t = a.T[tile_index(a)];
      CellPos c;
      c.pd = a.P[t.patch];
      const RhsConst& k = kl.k[c.pd.lev];
      const int tx = (int)threadIdx.x, ty = (int)threadIdx.y;
      const int nloc = min(TX, c.pd.nx - t.i0), mloc = min(TY, c.pd.ny - t.j0);
      c.i = t.i0 + tx;
      c.j = t.j0 + ty;
      c.k = t.k;
      c.st[0] = 1;
      c.st[1] = c.pd.sy;
      c.st[2] = c.pd.sz;
      c.c0 = c.pd.cell_off + (c.i + a.g) + (long long)(c.j + a.g) * c.pd.sy +
             (long long)(c.k + a.gz) * c.pd.sz;
      const long long c0 = c.c0, sy = c.st[1];
      if (tx < nloc && ty < mloc) {
         fx[ty][tx] = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, 0, c0 - 1, c0);
         fy[ty][tx] = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, 1, c0 - sy, c0);
      }
      // the faces closing the rows: one lane a row, all in the first wave; the
      // row closing the columns: the second wave
      if (ty == 0 && tx < mloc) {
         const long long e = c0 - tx + nloc + tx * sy;
         fx[tx][nloc] = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, 0, e - 1, e);
      }
      if (ty == 1 && tx < nloc) {
         const long long e = c0 + (long long)(mloc - 1) * sy;
         fy[mloc][tx] = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, 1, e - sy, e);
      }
      __syncthreads();
      if (tx >= nloc || ty >= mloc) return;
      double r = (fx[ty][tx + 1] - fx[ty][tx]) * k.dxinv[0];
      r = r + (fy[ty + 1][tx] - fy[ty][tx]) * k.dxinv[1];
      if (NDIM == 3) {
         const long long sz = c.st[2];
         double flo = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, 2, c0 - sz, c0);
         double fhi = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, 2, c0, c0 + sz);
         r = r + (fhi - flo) * k.dxinv[2];
      }
      rhs_tail<NDIM, FE, CONC, FIN>(a, p, k, c, r, phi, q, cc, cl, cs, gni, Dc, Dphi, yp, yq, yc, fin, iq,
                                    ic);
   } else {
      CellPos c;
      if (!cell_pos(a, 0, c)) return;
      const RhsConst& k = kl.k[c.pd.lev];
      const long long c0 = c.c0;
      double r = 0.0;
#pragma unroll
      for (int d = 0; d < NDIM; d++) {
         double flo = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, d, c0 - c.st[d], c0);
         double fhi = phase_face_flux<NDIM, FLUX>(p, k, phi, q, a.ncg, c.st, d, c0, c0 + c.st[d]);
         double dt = (fhi - flo) * k.dxinv[d];
         r = (d == 0) ? dt : r + dt;
      }
      rhs_tail<NDIM, FE, CONC, FIN>(a, p, k, c, r, phi, q, cc, cl, cs, gni, Dc, Dphi, yp, yq, yc, fin, iq,
                                    ic);
   }
}

}  // namespace

int launch_rhs_all(const Level& L, const ampe_model_params& p, const RhsLev& k, const double* y,
                   int iq, int ic, const double* cl, const double* cs, const double* gni,
                   double* Dc, double* Dphi, int conc, double* rhs, hipStream_t s, const KryFin* fin)
{
   const int fe = ic >= 0 ? p.fe_model : kFeNone;
   if (fin && conc != (ic >= 0 ? 1 : 0)) {
      set_error("rhs: a full evaluation's values, or an EBS composition's, are stored");
      return -1;
   }
   const KryFin kf = fin ? *fin : KryFin{};
   const double* q = iq >= 0 ? y + (long long)iq * L.ncg : nullptr;
   const double* cc = ic >= 0 ? y + (long long)ic * L.ncg : nullptr;
   double* yq = iq >= 0 ? rhs + (long long)iq * L.ncg : nullptr;
   double* yc = ic >= 0 ? rhs + (long long)ic * L.ncg : nullptr;
   const LevelArgs a = level_args(L);
   auto go2 = [&](auto nd, auto fl, auto f, auto cn, auto fi) {
      hipLaunchKernelGGL((k_rhs_all<decltype(nd)::value, decltype(fl)::value, decltype(f)::value,
                                    decltype(cn)::value, decltype(fi)::value>),
                         dim3(L.ncell_tiles), dim3(TX, TY), 0, s, a, p, k, y, q, cc, cl, cs, gni,
                         Dc, Dphi, rhs, yq, yc, kf, iq, ic);
   };
   auto go = [&](auto nd, auto fl, auto f, auto cn) {
      // (values are passed on by evaluations whose composition, if any, is formed here)
      if constexpr (decltype(cn)::value == (decltype(f)::value == kFeNone ? 0 : 1)) {
         if (fin) return go2(nd, fl, f, cn, std::true_type());
      }
      go2(nd, fl, f, cn, std::false_type());
   };
   using I0 = std::integral_constant<int, 0>;
   using I1 = std::integral_constant<int, 1>;
   using I2 = std::integral_constant<int, 2>;
   using I3 = std::integral_constant<int, 3>;
   auto by_conc = [&](auto nd, auto fl, auto f) {
      if (conc == 0)
         go(nd, fl, f, I0());
      else if (conc == 1)
         go(nd, fl, f, I1());
      else
         go(nd, fl, f, I2());
   };
   static_assert(AMPE_FE_QUADRATIC == 0 && AMPE_FE_CALPHAD_BINARY == 1 && AMPE_FE_KKS_DILUTE == 2,
                 "the dispatch below");
   auto by_fe = [&](auto nd, auto fl) {
      if (fe == AMPE_FE_QUADRATIC)
         by_conc(nd, fl, I0());
      else if (fe == AMPE_FE_CALPHAD_BINARY)
         by_conc(nd, fl, I1());
      else if (fe == AMPE_FE_KKS_DILUTE)
         by_conc(nd, fl, I2());
      else
         go(nd, fl, I3(), I0());
   };
   static_assert(AMPE_FLUX_SIMPLE == 0 && AMPE_FLUX_ISOTROPIC == 1 && AMPE_FLUX_ANISOTROPIC == 2,
                 "the dispatch below");
   if (L.ndim == 3) {
      if (p.flux_type == AMPE_FLUX_ANISOTROPIC)
         by_fe(I3(), I2());
      else
         by_fe(I3(), I0());
   } else if (p.flux_type == AMPE_FLUX_ANISOTROPIC) {
      by_fe(I2(), I2());
   } else if (p.flux_type == AMPE_FLUX_ISOTROPIC) {
      by_fe(I2(), I1());
   } else {
      by_fe(I2(), I0());
   }
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

}  // namespace ampe
