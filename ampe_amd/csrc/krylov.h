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

// work2 = sig (z h) + ycur
int kry_mid(const Level& L, int nc, double sig, const double* z, double h, const double* ycur,
            double* work2, hipStream_t s);
// v = z h + (-gamma) (siginv jv + (-siginv) fcur), written as pin says; with
// pin.f out may be null.
int kry_finish(const Level& L, int nc, double siginv, double gamma, const double* z, double h,
               const double* jv, const double* fcur, double* out, const PrecIn& pin,
               hipStream_t s);
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
