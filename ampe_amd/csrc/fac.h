// FAC preconditioner launch interface (see fac.hip).
#pragma once

#include "kernels.h"

namespace ampe {

// A u = M div(D grad u) + C u; a NULL field pointer selects the constant.
template <typename T>
struct EllOp {
   const T* D = nullptr;
   T Dc = 0;
   const T* C = nullptr;
   T Cc = 0;
   const T* M = nullptr;
   T Mc = 0;
};

// Preconditioner blocks that are swept together: each slot holds components
// [comp, comp + ncomp) of the shared right-hand side and solution vectors and
// their operator; a kernel over a set runs all slots in one launch.
template <typename T>
struct SweepSlot {
   int kind = 0;  // 0 elliptic (op), 1 orientation (face coefficients D, sm, gamma)
   int comp = 0, ncomp = 1;
   const T* D = nullptr;
   T Dc = 0;
   const T* C = nullptr;
   T Cc = 0;
   const T* M = nullptr;
   T Mc = 0;
   const T* sm = nullptr;
   T gamma = 0;
   const T* b = nullptr;  // the slot's own right-hand side instead of the shared one's components
};
// How a set's vectors are stored and read: split: the row parity-split layout
// (every component; coefficients natural); wrap: neighbours across the
// boundary of a one-patch periodic level read in place (level_wrap_ok), no
// ghost filled; from 1 / 2: the first red / black colour of a solve from zero
// (checker_ok levels).
struct SetForm {
   bool split = false, wrap = false;
   int from = 0;
};
// The split layout is the FP32 vectors'.
template <typename T>
constexpr bool kCanSplit = false;
template <>
inline constexpr bool kCanSplit<float> = true;
// Calls f with split as std::integral_constant, where the element type has it; -1
// where it has not.
template <typename T, class F>
int split_dispatch(bool split, F&& f)
{
   if constexpr (kCanSplit<T>) {
      if (split) {
         f(std::true_type());
         return 0;
      }
   } else if (split) {
      set_error("the row parity-split layout is for FP32 vectors");
      return -1;
   }
   f(std::false_type());
   return 0;
}
constexpr int kMaxSlots = 16;
template <typename T>
struct SweepSet {
   int n = 0;
   SweepSlot<T> s[kMaxSlots];
};
// Appends ncomp components sharing one operator, elliptic ones four to a slot
// (their coefficients are read once for the four); -1 when no slot is left.
template <typename T>
int sweep_add(SweepSet<T>& set, const SweepSlot<T>& proto, int comp, int ncomp);

// One colour of every slot's red-black sweep, and every slot's residual.
template <typename T>
int launch_set_sweep(const Level& L, const SweepSet<T>& set, const double* dx, const T* rhs, T* x,
                     int color, const SetForm& form, hipStream_t s);
template <typename T>
int launch_set_residual(const Level& L, const SweepSet<T>& set, const double* dx, const T* rhs,
                        const T* x, T* res, bool split, hipStream_t s);
// b (on coarse, the fine boxes halved) = the restriction of every slot's
// residual on fine after sweeps that end with the black colour: the red cells'
// residuals alone (the caller checks red_residual_ok).
template <typename T>
int launch_set_resrestrict(const Level& coarse, const Level& fine, const SweepSet<T>& set,
                           const double* dx, const T* rhs, const T* x, T* b, const SetForm& form,
                           hipStream_t s);
// Algorithmic bytes of one colour of a set's sweep: all solution values read
// and the colour's written, the colour's right-hand sides, the face and cell
// coefficients read once.
template <typename T>
double set_sweep_bytes(const Level& L, const SweepSet<T>& set, int from)
{
   const double n = (double)L.ncell;
   double v = 0.0;
   for (int i = 0; i < set.n; i++) {
      const SweepSlot<T>& o = set.s[i];
      // the first red colour reads no solution value, the first black one the
      // red half only
      const double read = from == 0 ? 1.0 : (from == 1 ? 0.0 : 0.5);
      v += o.ncomp * n * (read + 0.5 + 0.5);
      if (o.D) v += (double)L.nside_tot;
      v += n * ((o.C != nullptr) + (o.M != nullptr) + (o.sm != nullptr));
   }
   return v * sizeof(T);
}

int launch_phase_C(const Level& L, const ampe_model_params& p, double gamma,
                   const double* phi, const double* M, double* C, hipStream_t s);

// One colour sweep; with want_max the per-tile max |res| lands in L.partial.
template <typename T>
int launch_rbgs(const Level& L, const EllOp<T>& op, const double* dx, const T* rhs, T* u,
                int color, bool want_max, hipStream_t s);

// res = rhs - A u; if part is not null the per-tile sum res^2 lands in
// part[0 .. L.ncell_tiles).
template <typename T>
int launch_residual(const Level& L, const EllOp<T>& op, const double* dx, const T* rhs,
                    const T* u, T* res, double* part, hipStream_t s);

// Orientation block: one colour of the red-black sweep, and the residual
// (split: rhs, z and res in the row parity-split layout).
template <typename T>
int launch_quat_rbgs(const Level& L, const T* fc, const T* sm, double gamma, const double* dx,
                     int ncomp, const T* rhs, T* z, int color, hipStream_t s);

template <typename T>
int launch_quat_residual(const Level& L, const T* fc, const T* sm, double gamma,
                         const double* dx, int ncomp, const T* rhs, const T* z, T* res,
                         double* part, hipStream_t s, bool split = false);

// launch_set_resrestrict of one elliptic block, and of one orientation block
// of one, two or four components.
template <typename T>
int launch_ell_resrestrict(const Level& coarse, const Level& fine, const EllOp<T>& op,
                           const double* dx, const T* rhs, const T* u, T* b, hipStream_t s);
template <typename T>
int launch_quat_resrestrict(const Level& coarse, const Level& fine, const T* fc, const T* sm,
                            double gamma, const double* dx, int ncomp, const T* rhs, const T* z,
                            T* b, hipStream_t s);

// ------------------------------------------------------------ vectors
// Flat element-wise ops over n entries (whole ghosted vectors).
// One red-black sweep of the orientation block from zin (ghosts filled) into
// zout in one pass (plus a ghost fill of zout and a pass over the patches'
// outer layer): the values of the red launch followed by the black launch.
template <typename T>
int launch_quat_rbgs_fused(const Level& L, const T* fc, const T* sm, double gamma,
                           const double* dx, int ncomp, const T* rhs, const T* zin, T* zout,
                           hipStream_t s);
int vec_axpby(long long n, double a, const double* x, double b, const double* y, double* z,
              hipStream_t s);
int vec_fill(long long n, double v, double* z, hipStream_t s);
int vec_mul(long long n, const double* x, const double* y, double* z, hipStream_t s);
int vec_div(long long n, const double* x, const double* y, double* z, hipStream_t s);
int vec_ewt(long long n, const double* y, double rtol, double atol, double* w, hipStream_t s);
int vec_bdf2_hist(long long n, double c1, const double* y, double c2, const double* yp,
                  double* out, hipStream_t s);
int vec_to_f32(long long n, const double* x, float* y, hipStream_t s);
int vec_axpby_f(long long n, float* u, const float* e, hipStream_t s);  // u += e
// z[0, n) = 0 by a kernel (usable under HIP graph capture)
template <typename T>
int fill_zero(T* z, long long n, hipStream_t s);
int vec_to_f64(long long n, const float* x, double* y, hipStream_t s);
int vec_div_f(long long n, const double* x, const double* sm, double* y, hipStream_t s);
int vec_sqrt(long long n, const double* x, double* y, hipStream_t s);
// Preconditioner input / output over nc component blocks (orientation blocks
// [iq, iq+ql) scaled by 1/sqrt(M) on input, sqrt(M) on output); u, when given,
// is zeroed by psolve_in.  With f null (FP64) only the orientation blocks go to
// fq.  split (a level): the blocks from component sp0 on are stored in that
// level's row parity-split layout.
template <typename T>
int psolve_in(long long ng, int nc, int iq, int ql, const double* r, const double* sm, T* f,
              T* fq, T* u, hipStream_t s, const Level* split = nullptr, int sp0 = 0);
template <typename T>
int psolve_out(long long ng, int nc, int iq, int ql, const T* u, const double* sm,
               double* z, hipStream_t s, const Level* split = nullptr, int sp0 = 0);
int vec_scale_comp(long long ng, int ncomp, const double* sm, double* x, hipStream_t s);
// Reductions over interior cells of ncomp component blocks (host result,
// synchronises s).
int vec_dot(const Level& L, int ncomp, const double* x, const double* y, double* out,
            hipStream_t s);
int vec_sumsq_w(const Level& L, int ncomp, const double* x, const double* w, double* out,
                hipStream_t s);

}  // namespace ampe
