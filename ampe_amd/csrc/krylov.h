// Fused Newton-Krylov vector kernels (see krylov.hip).  Host results of the
// reductions are raw sums over interior cells (no cell-volume factor).
#pragma once

#include "kernels.h"

namespace ampe {

constexpr int kMaxKrylov = 32;

// How a preconditioner right-hand side r is written: the orientation components
// [iq, iq + ql) divided by sqrt(M) = sm (null: none), and with f in FP32 to f.
struct PrecIn {
   float* f = nullptr;
   const double* sm = nullptr;
   int iq = 0, ql = 0;
   int sp0 = 1 << 30;  // components of f from sp0 on are in the row parity-split layout
};

// A preconditioned vector as the solve left it: FP32 u, or FP64 z; orientation
// components to be multiplied by sm (null: none).
struct PrecOut {
   const float* u = nullptr;
   const double* z = nullptr;
   const double* sm = nullptr;
   int iq = 0, ql = 0;
   int sp0 = 1 << 30;  // components of u from sp0 on are in the row parity-split layout
};

// Basis vectors (not scaled by ewt, not normalised) and a factor for each.
struct VecList {
   int n;
   const double* v[kMaxKrylov];
   double y[kMaxKrylov];
};

// What makes the next preconditioner right-hand side of a difference quotient's
// jv: v = z h + (-gamma) (siginv jv + (-siginv) f), written to out and as pin says
// (with pin.f out may be null).
struct KryFin {
   const double* z = nullptr;
   double h = 0.0, siginv = 0.0, gamma = 0.0;
   const double* f = nullptr;
   double* out = nullptr;
   PrecIn pin;
};

__device__ __forceinline__ bool in_range(int m, int iq, int ql) { return m >= iq && m < iq + ql; }

__device__ __forceinline__ void prec_in(const LevelArgs& a, const PrecIn& pin, const CellPos& c,
                                        long long sp, int m, double v, double sm, double* out)
{
   if (pin.sm && in_range(m, pin.iq, pin.ql)) v = v / sm;
   if (out) out[m * a.ncg + c.c0] = v;
   if (pin.f) pin.f[m * a.ncg + (m >= pin.sp0 ? sp : c.c0)] = (float)v;
}

__device__ __forceinline__ double kry_fin(const KryFin& k, long long i, double jv)
{
   return k.z[i] * k.h + (-k.gamma) * (k.siginv * jv + (-k.siginv) * k.f[i]);
}

// work2 = sig (z h) + ycur; with ghosts also on the level's ghost cells, from the
// cells they copy.
int kry_mid(const Level& L, int nc, double sig, const double* z, double h, const double* ycur,
            double* work2, bool ghosts, hipStream_t s);
int kry_finish(const Level& L, int nc, const KryFin& fin, const double* jv, hipStream_t s);
// b = gamma f - (y - a), written as pin says (out may be null with pin.f).
int kry_newton_rhs(const Level& L, int nc, double gamma, const double* f, const double* y,
                   const double* ah, double* out, const PrecIn& pin, hipStream_t s);
// z = src, *sumsq = (ewt z) . (ewt z)
int kry_start(const Level& L, int nc, const PrecOut& src, const double* ewt, double* z,
              double* sumsq, hipStream_t s);
// z = src orthogonalised against the vectors of vl (vl.y: their normalisation
// factors) by classical (at most kMaxCgs - 1 vectors) or modified Gram-Schmidt in
// the ewt-weighted product.  sums[k] = src . v[k] of the products taken,
// sums[vl.n] = z . z, and with classical sums[vl.n + 1] = src . src.
constexpr int kMaxCgs = 16;
int kry_cgs(const Level& L, int nc, const PrecOut& src, const VecList& vl, double cv,
            const double* ewt, double* z, double* sums, hipStream_t s);
int kry_mgs(const Level& L, int nc, const PrecOut& src, const VecList& vl, double cv,
            const double* ewt, double* z, double* sums, hipStream_t s);
// x = sum_k vl.y[k] vl.v[k] (k in order); y = y + x; *sumsq = (ewt x) . (ewt x)
int kry_newton_update(const Level& L, int nc, const VecList& vl, const double* ewt, double* y,
                      double* sumsq, hipStream_t s);

}  // namespace ampe
