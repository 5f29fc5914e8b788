// FAC preconditioner kernels: phase operator coefficient C, red-black
// Gauss-Seidel colour sweeps and residuals of A u = M div(D grad u) + C u, and
// the orientation block's symmetrised operator I + gamma sqrt(M) L sqrt(M).
// Templated on the storage/compute type: double for the FP64 path, float for
// the mixed-precision preconditioner.
#include <type_traits>

#include "fac.h"

namespace ampe {

// PhaseFACOps::setCOnPatchPrivate (source/PhaseFACOps.cc:101-183)
__global__ void __launch_bounds__(256) k_phase_C(LevelArgs a, ampe_model_params p, double gamma,
                                                 const double* __restrict__ phi,
                                                 const double* __restrict__ M,
                                                 double* __restrict__ C)
{
   CellPos c;
   if (!cell_pos(a, 0, c)) return;
   double g2 = d2well(phi[c.c0], p.phi_well_type);
   double gm = gamma * (M ? M[c.c0] : p.phi_mobility);
   C[c.c0] = 1.0 + gm * p.phi_well_scale * g2;
}

// Colour of the update: efo_rbgswithfluxmax* walk row (j, k) from
// ifirst + ioffset in steps of 2, with ioffset = 1 when the parity of
// (jfirst + j) [2-D] or (ifirst + j + k) [3-D] differs from the colour
// (source/fortran/2d/ellipticfacops.m4:111-130, 3d/ellipticfacops.m4).
template <int NDIM>
__device__ __forceinline__ bool is_color(const CellPos& c, int color)
{
   int gj = c.pd.lo[1] + c.j;
   int x = (NDIM == 3) ? c.pd.lo[0] + gj + (c.pd.lo[2] + c.k) : c.pd.lo[1] + gj;
   int io = ((x - (x / 2) * 2) != color) ? 1 : 0;
   return ((c.i - io) & 1) == 0 && c.i >= io;
}

// Colour-compact mapping: a workgroup of TX/2 x TY threads covers one tile,
// each thread the one cell of the colour in its pair (2 tx, 2 tx + 1) of the
// row, so every lane updates a cell (the full-tile mapping leaves half of
// them idle).  Plane t.k + kk; false when outside the box.
template <int NDIM>
__device__ __forceinline__ bool cell_pos_color(const LevelArgs& a, int kk, int color,
                                               CellPos& c)
{
   const Tile t = a.T[tile_index(a)];
   c.pd = a.P[t.patch];
   c.j = t.j0 + (int)threadIdx.y;
   c.k = t.k + kk;
   int gj = c.pd.lo[1] + c.j;
   int x = (NDIM == 3) ? c.pd.lo[0] + gj + (c.pd.lo[2] + c.k) : c.pd.lo[1] + gj;
   int io = ((x - (x / 2) * 2) != color) ? 1 : 0;
   c.i = t.i0 + 2 * (int)threadIdx.x + io;  // t.i0 is a multiple of TX (even)
   if (c.i >= c.pd.nx || c.j >= c.pd.ny || c.k >= c.pd.nz) return false;
   c.st[0] = 1;
   c.st[1] = c.pd.sy;
   c.st[2] = c.pd.sz;
   c.c0 = c.pd.cell_off + (c.i + a.g) + (long long)(c.j + a.g) * c.pd.sy +
          (long long)(c.k + a.gz) * c.pd.sz;
   return true;
}

template <typename T>
struct OpArgs {
   const T* D;
   T Dc;
   const T* C;
   T Cc;
   const T* M;
   T Mc;
};

// res = rhs - M div(D grad u) - C u at one cell; *diag = M sum D/h^2 - C
// (the reciprocal is dudr of efo_rbgswithfluxmax*).
template <typename T, int NDIM>
__device__ __forceinline__ T op_residual(const LevelArgs& a, const CellPos& c, const OpArgs<T>& op,
                                         const T* __restrict__ rhs, const T* __restrict__ u,
                                         const T* dinv, T* diag)
{
   const long long c0 = c.c0;
   const int ijk[3] = {c.i, c.j, c.k};
   T div = 0, dsum = 0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      T dlo, dhi;
      if (op.D) {
         int lo[3] = {ijk[0], ijk[1], ijk[2]};
         long long flo = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
         lo[d] += 1;
         long long fhi = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
         dlo = op.D[flo];
         dhi = op.D[fhi];
      } else {
         dlo = dhi = op.Dc;
      }
      long long s = c.st[d];
      T flo = dinv[d] * dlo * (u[c0] - u[c0 - s]);
      T fhi = dinv[d] * dhi * (u[c0 + s] - u[c0]);
      T t = dinv[d] * (fhi - flo);
      T ds = dinv[d] * dinv[d] * (dhi + dlo);
      div = (d == 0) ? t : div + t;
      dsum = (d == 0) ? ds : dsum + ds;
   }
   T m = op.M ? op.M[c0] : op.Mc;
   T cc = op.C ? op.C[c0] : op.Cc;
   *diag = m * dsum - cc;
   return rhs[c0] - m * div - cc * u[c0];
}

template <typename T>
__device__ __forceinline__ void block_store_max(T v, double* partial)
{
   __shared__ double sh[TX * TY];
   int t = threadIdx.x + TX * threadIdx.y;
   sh[t] = (double)v;
   __syncthreads();
   for (int w = TX * TY / 2; w > 0; w >>= 1) {
      if (t < w) sh[t] = sh[t + w] > sh[t] ? sh[t + w] : sh[t];
      __syncthreads();
   }
   if (t == 0) partial[blockIdx.x] = sh[0];
}

template <typename T>
__device__ __forceinline__ void block_store_sum(double v, double* partial)
{
   __shared__ double sh[TX * TY];
   int t = threadIdx.x + TX * threadIdx.y;
   sh[t] = v;
   __syncthreads();
   for (int w = TX * TY / 2; w > 0; w >>= 1) {
      if (t < w) sh[t] = sh[t] + sh[t + w];
      __syncthreads();
   }
   if (t == 0) partial[blockIdx.x] = sh[0];
}

// One colour of efo_rbgswithfluxmax{var,con}dc{var,con}sf
// (source/fortran/2d/ellipticfacops.m4:60-345): u += -res * dudr.
template <typename T, int NDIM>
__device__ __forceinline__ T rbgs_cell(const LevelArgs& a, const CellPos& c, const OpArgs<T>& op,
                                       const T* dinv, const T* __restrict__ rhs, T* __restrict__ u)
{
   T diag;
   T res = op_residual<T, NDIM>(a, c, op, rhs, u, dinv, &diag);
   T dudr = T(1) / diag;
   T du = -res * dudr;
   u[c.c0] = u[c.c0] + du * T(1);
   return res < 0 ? -res : res;
}

template <typename T, int NDIM>
__global__ void __launch_bounds__(256) k_rbgs(LevelArgs a, OpArgs<T> op, T di0, T di1, T di2,
                                              const T* __restrict__ rhs, T* __restrict__ u,
                                              int color, double* __restrict__ partial)
{
   T absres = 0;
   const T dinv[3] = {di0, di1, di2};
   AMPE_COLUMN_BEGIN(a, c)
   if (!is_color<NDIM>(c, color)) continue;
   T ar = rbgs_cell<T, NDIM>(a, c, op, dinv, rhs, u);
   absres = ar > absres ? ar : absres;
   AMPE_COLUMN_END
   if (partial) block_store_max<T>(absres, partial);
}

// efo_compres*sca (source/fortran/2d/ellipticfacops.m4:346-446) + sum res^2
template <typename T, int NDIM>
__global__ void __launch_bounds__(256) k_residual(LevelArgs a, OpArgs<T> op, T di0, T di1, T di2,
                                                  const T* __restrict__ rhs, const T* __restrict__ u,
                                                  T* __restrict__ res, double* __restrict__ partial)
{
   double sq = 0.0;
   AMPE_COLUMN_BEGIN(a, c)
   T dinv[3] = {di0, di1, di2};
   T diag;
   T r = op_residual<T, NDIM>(a, c, op, rhs, u, dinv, &diag);
   res[c.c0] = r;
   sq += (double)r * (double)r;
   AMPE_COLUMN_END
   if (partial) block_store_sum<T>(sq, partial);
}

// ------------------------------------------------------------ orientation
// Row of A = I + gamma sqrt(M) L sqrt(M), L from face coefficients:
// off-diagonal fc/h^2, diagonal -sum fc/h^2 (set_j_ij2d/3d, set_stencil2d/3d,
// source/fortran/2d/quatlevelsolver.m4:9-120).  Returns A z at one cell for
// component block zc and the centre coefficient.
template <typename T, int NDIM>
__device__ __forceinline__ T quat_row(const LevelArgs& a, const CellPos& c, const T* __restrict__ fc,
                                      const T* __restrict__ sm, T gamma, const T* hinv2,
                                      const T* __restrict__ z, T* center);

// The same row with the z values supplied by zv(d, side): the cell itself for
// d < 0, else its neighbour across the low (side -1) or high (+1) face of
// direction d.  Same operations in the same order as quat_row.
template <typename T, int NDIM, class ZV>
__device__ __forceinline__ T quat_row_zv(const LevelArgs& a, const CellPos& c,
                                         const T* __restrict__ fc, const T* __restrict__ sm,
                                         T gamma, const T* hinv2, const ZV& zv, T* center)
{
   const long long c0 = c.c0;
   const int ijk[3] = {c.i, c.j, c.k};
   T olo[3], ohi[3];
   T diag = 0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      int lo[3] = {ijk[0], ijk[1], ijk[2]};
      long long flo = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      lo[d] += 1;
      long long fhi = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      olo[d] = fc[flo] * hinv2[d];
      ohi[d] = fc[fhi] * hinv2[d];
      diag = (d == 0) ? -olo[0] - ohi[0] : diag - olo[d] - ohi[d];
   }
   T fac = gamma * sm[c0];
   *center = fac * diag * sm[c0] + T(1);
   T r = *center * zv(-1, 0);
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      long long s = c.st[d];
      r = r + fac * olo[d] * sm[c0 - s] * zv(d, -1) + fac * ohi[d] * sm[c0 + s] * zv(d, 1);
   }
   return r;
}

template <typename T, int NDIM>
__device__ __forceinline__ T quat_row(const LevelArgs& a, const CellPos& c, const T* __restrict__ fc,
                                      const T* __restrict__ sm, T gamma, const T* hinv2,
                                      const T* __restrict__ z, T* center)
{
   const long long c0 = c.c0;
   const int ijk[3] = {c.i, c.j, c.k};
   T olo[3], ohi[3];
   T diag = 0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      int lo[3] = {ijk[0], ijk[1], ijk[2]};
      long long flo = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      lo[d] += 1;
      long long fhi = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      olo[d] = fc[flo] * hinv2[d];
      ohi[d] = fc[fhi] * hinv2[d];
      diag = (d == 0) ? -olo[0] - ohi[0] : diag - olo[d] - ohi[d];
   }
   T fac = gamma * sm[c0];
   *center = fac * diag * sm[c0] + T(1);
   T r = *center * z[c0];
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      long long s = c.st[d];
      r = r + fac * olo[d] * sm[c0 - s] * z[c0 - s] + fac * ohi[d] * sm[c0 + s] * z[c0 + s];
   }
   return r;
}

// The row's coefficients at one cell, shared by every component: centre
// gamma sm^2 diag + 1 and the neighbour weights gamma sm fc/h^2 sm_nbr (the
// products quat_row forms, in its order).
template <typename T>
struct QuatRowCoef {
   T center;
   T wlo[3], whi[3];
};

template <typename T, int NDIM>
__device__ __forceinline__ QuatRowCoef<T> quat_row_coef(const LevelArgs& a, const CellPos& c,
                                                        const T* __restrict__ fc,
                                                        const T* __restrict__ sm, T gamma,
                                                        const T* hinv2)
{
   const long long c0 = c.c0;
   const int ijk[3] = {c.i, c.j, c.k};
   T olo[3], ohi[3];
   T diag = 0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      int lo[3] = {ijk[0], ijk[1], ijk[2]};
      long long flo = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      lo[d] += 1;
      long long fhi = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
      olo[d] = fc[flo] * hinv2[d];
      ohi[d] = fc[fhi] * hinv2[d];
      diag = (d == 0) ? -olo[0] - ohi[0] : diag - olo[d] - ohi[d];
   }
   QuatRowCoef<T> w;
   T fac = gamma * sm[c0];
   w.center = fac * diag * sm[c0] + T(1);
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      w.wlo[d] = fac * olo[d] * sm[c0 - c.st[d]];
      w.whi[d] = fac * ohi[d] * sm[c0 + c.st[d]];
   }
   return w;
}

// Component values of one cell's row: the cell and its face neighbours.
template <typename T, int NDIM>
struct QuatRowVals {
   T zc, zl[NDIM], zh[NDIM];
};

// Where one cell's component values sit: the cell and its two neighbours in
// the row (rows above and below, planes before and after: the cell's index
// -+ the row / plane stride).  SPLIT: the row parity-split layout.
struct QuatIdx {
   long long c, xl, xh;
};

template <bool SPLIT>
__device__ __forceinline__ QuatIdx quat_idx(const LevelArgs& a, const CellPos& c)
{
   if (SPLIT) return {split_at(a, c, 0), split_at(a, c, -1), split_at(a, c, 1)};
   return {c.c0, c.c0 - 1, c.c0 + 1};
}

template <typename T, int NDIM>
__device__ __forceinline__ void quat_row_load(const CellPos& c, const QuatIdx& q,
                                              const T* __restrict__ zm, QuatRowVals<T, NDIM>& v)
{
   v.zc = zm[q.c];
   v.zl[0] = zm[q.xl];
   v.zh[0] = zm[q.xh];
#pragma unroll
   for (int d = 1; d < NDIM; d++) {
      v.zl[d] = zm[q.c - c.st[d]];
      v.zh[d] = zm[q.c + c.st[d]];
   }
}

// A z from the loaded values: the sum quat_row forms, in its order.
template <typename T, int NDIM>
__device__ __forceinline__ T quat_row_apply(const QuatRowCoef<T>& w, const QuatRowVals<T, NDIM>& v)
{
   T r = w.center * v.zc;
#pragma unroll
   for (int d = 0; d < NDIM; d++) r = r + w.wlo[d] * v.zl[d] + w.whi[d] * v.zh[d];
   return r;
}

// ------------------------------------------------------------ fused sweep
// One red-black sweep of the orientation block in one pass, zin -> zout
// (zin ghost-filled, not written).  A workgroup first updates every red cell
// of its tile grown by one cell in each direction (neighbouring tiles'
// cells included, from zin only) into LDS, then the black cells of its tile
// from those red values: the same operations as the red launch followed by
// the black launch, so the same values, with zin read once instead of twice.
// Black cells on a patch's outer layer need values of ghost cells; they keep
// their previous value here and are updated by k_quat_rbgs_shell after a
// ghost fill of zout.
constexpr int kRX = TX + 2, kRY = TY + 2;

template <int NDIM>
__device__ __forceinline__ void make_cell(const LevelArgs& a, const PatchDev& pd, int i, int j,
                                          int k, CellPos& c)
{
   c.pd = pd;
   c.i = i;
   c.j = j;
   c.k = k;
   c.st[0] = 1;
   c.st[1] = pd.sy;
   c.st[2] = pd.sz;
   c.c0 = pd.cell_off + (i + a.g) + (long long)(j + a.g) * pd.sy + (long long)(k + a.gz) * pd.sz;
}

template <int NDIM>
__device__ __forceinline__ bool outer_layer(const CellPos& c)
{
   return c.i == 0 || c.i == c.pd.nx - 1 || c.j == 0 || c.j == c.pd.ny - 1 ||
          (NDIM == 3 && (c.k == 0 || c.k == c.pd.nz - 1));
}

template <typename T, int NDIM>
__global__ void __launch_bounds__(256) k_quat_rbgs_fused(LevelArgs a, const T* __restrict__ fc,
                                                         const T* __restrict__ sm, T gamma,
                                                         T hi0, T hi1, T hi2, int ncomp,
                                                         const T* __restrict__ rhs,
                                                         const T* __restrict__ zin,
                                                         T* __restrict__ zout)
{
   // a column of the tile's planes [t.k, kend): the red values of the tile
   // grown by one cell in x and y for planes k-1, k, k+1 live in a ring of
   // three LDS slots (slot = plane % 3); each step adds plane k+1, then
   // updates the black cells of plane k
   constexpr int NP = kRX * kRY;
   constexpr int RING = NDIM == 3 ? 3 : 1;
   __shared__ T red[RING][4][NP];
   const T hinv2[3] = {hi0, hi1, hi2};
   const Tile t = a.T[tile_index(a)];
   const PatchDev pd = a.P[t.patch];
   const int kend = NDIM == 3 ? min(t.k + a.nz_tile, pd.nz) : 1;
   const int tid = (int)threadIdx.x + TX * (int)threadIdx.y;
   auto red_plane = [&](int p) {
      if (p < 0 || p >= pd.nz) return;
      const int slot = NDIM == 3 ? p % 3 : 0;
      for (int r = tid; r < NP; r += TX * TY) {
         const int ri = r % kRX - 1, rj = r / kRX - 1;
         const int i = t.i0 + ri, j = t.j0 + rj;
         if (i < 0 || i >= pd.nx || j < 0 || j >= pd.ny) continue;
         CellPos c;
         make_cell<NDIM>(a, pd, i, j, p, c);
         if (!is_color<NDIM>(c, 0)) continue;
         const bool own = ri >= 0 && ri < TX && rj >= 0 && rj < TY && p >= t.k && p < kend;
         for (int m = 0; m < ncomp; m++) {
            const T* zm = zin + m * a.ncg;
            T center;
            T az = quat_row<T, NDIM>(a, c, fc, sm, gamma, hinv2, zm, &center);
            T res = rhs[m * a.ncg + c.c0] - az;
            T v = zm[c.c0] + res / center;
            red[slot][m][r] = v;
            if (own) zout[m * a.ncg + c.c0] = v;
         }
      }
   };
   if (NDIM == 3) red_plane(t.k - 1);
   red_plane(t.k);
   const int tx = (int)threadIdx.x, ty = (int)threadIdx.y;
   const int i = t.i0 + tx, j = t.j0 + ty;
   const int r0 = (tx + 1) + kRX * (ty + 1);
   for (int k = t.k; k < kend; k++) {
      if (NDIM == 3) red_plane(k + 1);
      __syncthreads();
      if (i < pd.nx && j < pd.ny) {
         CellPos c;
         make_cell<NDIM>(a, pd, i, j, k, c);
         if (!is_color<NDIM>(c, 0)) {
            if (outer_layer<NDIM>(c)) {
               // previous value for now: the ghost fill of zout then gives
               // every ghost cell the value the black launch would read (red
               // updated, black not; ghost sources lie on their patches' outer
               // layers, and in 2-D the colouring is per patch, so a neighbour
               // across a patch face can be black)
               for (int m = 0; m < ncomp; m++) zout[m * a.ncg + c.c0] = zin[m * a.ncg + c.c0];
            } else {
               const int s0 = NDIM == 3 ? k % 3 : 0;
               const int sm1 = NDIM == 3 ? (k + 2) % 3 : 0, sp1 = NDIM == 3 ? (k + 1) % 3 : 0;
               for (int m = 0; m < ncomp; m++) {
                  const T* zm = zin + m * a.ncg;
                  auto zv = [&](int d, int side) -> T {
                     if (d < 0) return zm[c.c0];
                     if (d == 0) return red[s0][m][r0 + side];
                     if (d == 1) return red[s0][m][r0 + side * kRX];
                     return red[side < 0 ? sm1 : sp1][m][r0];
                  };
                  T center;
                  T az = quat_row_zv<T, NDIM>(a, c, fc, sm, gamma, hinv2, zv, &center);
                  T res = rhs[m * a.ncg + c.c0] - az;
                  zout[m * a.ncg + c.c0] = zm[c.c0] + res / center;
               }
            }
         }
      }
      __syncthreads();
   }
}

// Black cells on the outer layer: neighbours from zout (ghost-filled: red
// cells updated, black cells still previous), own previous value from zin.
template <typename T, int NDIM>
__global__ void __launch_bounds__(256) k_quat_rbgs_shell(LevelArgs a, const T* __restrict__ fc,
                                                         const T* __restrict__ sm, T gamma,
                                                         T hi0, T hi1, T hi2, int ncomp,
                                                         const T* __restrict__ rhs,
                                                         const T* __restrict__ zin,
                                                         T* __restrict__ zout)
{
   CellPos c;
   if (!cell_pos(a, 0, c)) return;
   if (is_color<NDIM>(c, 0) || !outer_layer<NDIM>(c)) return;
   const T hinv2[3] = {hi0, hi1, hi2};
   for (int m = 0; m < ncomp; m++) {
      const T* zm = zin + m * a.ncg;
      const T* zo = zout + m * a.ncg;
      auto zv = [&](int d, int side) -> T {
         return d < 0 ? zm[c.c0] : zo[c.c0 + side * c.st[d]];
      };
      T center;
      T az = quat_row_zv<T, NDIM>(a, c, fc, sm, gamma, hinv2, zv, &center);
      T res = rhs[m * a.ncg + c.c0] - az;
      zout[m * a.ncg + c.c0] = zm[c.c0] + res / center;
   }
}

// Residual of one cell, every component (QL > 0: all loads of QL components
// before the first of them is used); returns the sum of the squared residuals
// (double).
template <typename T, int NDIM, int QL, bool SPLIT>
__device__ __forceinline__ double quat_residual_cell(const LevelArgs& a, const CellPos& c,
                                                     const T* __restrict__ fc,
                                                     const T* __restrict__ sm, T gamma,
                                                     const T* hinv2, int ncomp,
                                                     const T* __restrict__ rhs,
                                                     const T* __restrict__ z,
                                                     T* __restrict__ res)
{
   double sq = 0.0;
   const QuatRowCoef<T> w = quat_row_coef<T, NDIM>(a, c, fc, sm, gamma, hinv2);
   const QuatIdx q = quat_idx<SPLIT>(a, c);
   if (QL > 0) {
      QuatRowVals<T, NDIM> v[QL > 0 ? QL : 1];
      T rv[QL > 0 ? QL : 1];
#pragma unroll
      for (int m = 0; m < QL; m++) {
         quat_row_load<T, NDIM>(c, q, z + m * a.ncg, v[m]);
         rv[m] = rhs[m * a.ncg + q.c];
      }
#pragma unroll
      for (int m = 0; m < QL; m++) {
         T r = rv[m] - quat_row_apply<T, NDIM>(w, v[m]);
         res[m * a.ncg + q.c] = r;
         sq += (double)r * (double)r;
      }
   } else {
      for (int m = 0; m < ncomp; m++) {
         QuatRowVals<T, NDIM> v;
         quat_row_load<T, NDIM>(c, q, z + m * a.ncg, v);
         T r = rhs[m * a.ncg + q.c] - quat_row_apply<T, NDIM>(w, v);
         res[m * a.ncg + q.c] = r;
         sq += (double)r * (double)r;
      }
   }
   return sq;
}

template <typename T, int NDIM, int QL, bool SPLIT>
__global__ void __launch_bounds__(256) k_quat_residual(LevelArgs a, const T* __restrict__ fc,
                                                       const T* __restrict__ sm, T gamma, T hi0,
                                                       T hi1, T hi2, int ncomp,
                                                       const T* __restrict__ rhs,
                                                       const T* __restrict__ z, T* __restrict__ res,
                                                       double* __restrict__ partial)
{
   double sq = 0.0;
   const T hinv2[3] = {hi0, hi1, hi2};
   AMPE_COLUMN_BEGIN(a, c)
   sq += quat_residual_cell<T, NDIM, QL, SPLIT>(a, c, fc, sm, gamma, hinv2, ncomp, rhs, z, res);
   AMPE_COLUMN_END
   if (partial) block_store_sum<T>(sq, partial);
}

// ------------------------------------------------------------ block sets
// The elliptic row's coefficients at one cell, shared by the slot's
// components: dinv D of the low and high faces, M, C and the diagonal (the
// products op_residual forms, in its order).
template <typename T>
struct EllRowCoef {
   T wlo[3], whi[3], m, cc, diag;
};

template <typename T, int NDIM>
__device__ __forceinline__ EllRowCoef<T> ell_row_coef(const LevelArgs& a, const CellPos& c,
                                                      const SweepSlot<T>& o, const T* dinv)
{
   const int ijk[3] = {c.i, c.j, c.k};
   EllRowCoef<T> w;
   T dsum = 0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      T dlo, dhi;
      if (o.D) {
         int lo[3] = {ijk[0], ijk[1], ijk[2]};
         long long flo = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
         lo[d] += 1;
         long long fhi = face_idx(a, c.pd, d, lo[0], lo[1], lo[2]);
         dlo = o.D[flo];
         dhi = o.D[fhi];
      } else {
         dlo = dhi = o.Dc;
      }
      w.wlo[d] = dinv[d] * dlo;
      w.whi[d] = dinv[d] * dhi;
      T ds = dinv[d] * dinv[d] * (dhi + dlo);
      dsum = (d == 0) ? ds : dsum + ds;
   }
   w.m = o.M ? o.M[c.c0] : o.Mc;
   w.cc = o.C ? o.C[c.c0] : o.Cc;
   w.diag = w.m * dsum - w.cc;
   return w;
}

// rhs - A u of one component from the row's coefficients (op_residual's
// operations in its order).
template <typename T, int NDIM>
__device__ __forceinline__ T ell_row_residual(const EllRowCoef<T>& w, const T* dinv, T rhs,
                                              const QuatRowVals<T, NDIM>& v)
{
   T div = 0;
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      T flo = w.wlo[d] * (v.zc - v.zl[d]);
      T fhi = w.whi[d] * (v.zh[d] - v.zc);
      T t = dinv[d] * (fhi - flo);
      div = (d == 0) ? t : div + t;
   }
   return rhs - w.m * div - w.cc * v.zc;
}

// Where a cell and its face neighbours sit in one component block.  SPLIT: the
// row parity-split layout.  WRAP: the one patch of a periodic level, whose
// neighbours across the boundary are read where they are, at the patch's
// other side, so that no ghost is filled between two colours (the colours
// meet across the boundary as inside: the caller checks that the extents are
// even).
template <int NDIM>
struct NbrIdx {
   long long c, l[NDIM], h[NDIM];
};

template <int NDIM, bool SPLIT, bool WRAP>
__device__ __forceinline__ NbrIdx<NDIM> nbr_idx(const LevelArgs& a, const CellPos& c)
{
   NbrIdx<NDIM> q;
   const int nx = c.pd.nx, ig = c.i + a.g;
   const int il = (WRAP && c.i == 0) ? ig + nx - 1 : ig - 1;
   const int ih = (WRAP && c.i == nx - 1) ? ig - nx + 1 : ig + 1;
   const long long row = c.c0 - ig;
   q.c = SPLIT ? row + split_col(ig, c.pd.sy) : c.c0;
   q.l[0] = SPLIT ? row + split_col(il, c.pd.sy) : row + il;
   q.h[0] = SPLIT ? row + split_col(ih, c.pd.sy) : row + ih;
   const int ijk[3] = {c.i, c.j, c.k}, n[3] = {nx, c.pd.ny, c.pd.nz};
#pragma unroll
   for (int d = 1; d < NDIM; d++) {
      const long long s = c.st[d], w = (long long)(n[d] - 1) * s;
      q.l[d] = (WRAP && ijk[d] == 0) ? q.c + w : q.c - s;
      q.h[d] = (WRAP && ijk[d] == n[d] - 1) ? q.c - w : q.c + s;
   }
   return q;
}

template <typename T, int NDIM>
__device__ __forceinline__ void nbr_load(const NbrIdx<NDIM>& q, const T* __restrict__ x,
                                         QuatRowVals<T, NDIM>& v)
{
#pragma unroll
   for (int d = 0; d < NDIM; d++) {
      v.zl[d] = x[q.l[d]];
      v.zh[d] = x[q.h[d]];
   }
}

// Values of a component at the start of a sweep: FROM 0 any, 1 the whole
// field is zero (a red cell of a solve from zero), 2 the cell itself is zero
// (a black one after it).
template <typename T, int NDIM, int FROM>
__device__ __forceinline__ void nbr_start(const NbrIdx<NDIM>& q, const T* __restrict__ x,
                                          QuatRowVals<T, NDIM>& v)
{
   v.zc = FROM == 0 ? x[q.c] : T(0);
   if (FROM == 1) {
#pragma unroll
      for (int d = 0; d < NDIM; d++) v.zl[d] = v.zh[d] = T(0);
   } else {
      nbr_load<T, NDIM>(q, x, v);
   }
}

// Gauss-Seidel update of the orientation block at one cell: QL > 0 all loads
// of QL components before the first update, QL = 0 one component after the
// other.
template <typename T, int NDIM, int QL, int FROM>
__device__ __forceinline__ void set_quat_cell(const QuatRowCoef<T>& w, const NbrIdx<NDIM>& q,
                                              long long ncg, int ncomp,
                                              const T* __restrict__ b, T* __restrict__ x)
{
   if (QL > 0) {
      QuatRowVals<T, NDIM> v[QL > 0 ? QL : 1];
      T rv[QL > 0 ? QL : 1];
#pragma unroll
      for (int m = 0; m < QL; m++) {
         nbr_start<T, NDIM, FROM>(q, x + m * ncg, v[m]);
         rv[m] = b[m * ncg + q.c];
      }
#pragma unroll
      for (int m = 0; m < QL; m++) {
         T res = FROM == 1 ? rv[m] : rv[m] - quat_row_apply<T, NDIM>(w, v[m]);
         x[m * ncg + q.c] = v[m].zc + res / w.center;
      }
      return;
   }
   for (int m = 0; m < ncomp; m++) {
      QuatRowVals<T, NDIM> v;
      nbr_start<T, NDIM, FROM>(q, x + m * ncg, v);
      T res = b[m * ncg + q.c];
      if (FROM != 1) res = res - quat_row_apply<T, NDIM>(w, v);
      x[m * ncg + q.c] = v.zc + res / w.center;
   }
}

// One colour's update of slot o at cell c.  KIND: the slot's kind, QL: the
// orientation components taken at once; KIND < 0: the slot's own, four at once or
// one after the other.
template <typename T, int NDIM, bool SPLIT, bool WRAP, int FROM, int KIND, int QL>
__device__ __forceinline__ void sweep_slot(const LevelArgs& a, const CellPos& c,
                                           const SweepSlot<T>& o, const T* dinv, const T* hinv2,
                                           const T* __restrict__ rhs, T* __restrict__ x)
{
   const T* b = o.b ? o.b : rhs + o.comp * a.ncg;
   T* u = x + o.comp * a.ncg;
   const NbrIdx<NDIM> q = nbr_idx<NDIM, SPLIT, WRAP>(a, c);
   if (KIND < 0 ? o.kind == 1 : KIND == 1) {
      const QuatRowCoef<T> w = quat_row_coef<T, NDIM>(a, c, o.D, o.sm, o.gamma, hinv2);
      if (KIND >= 0)
         set_quat_cell<T, NDIM, QL, FROM>(w, q, a.ncg, o.ncomp, b, u);
      else if (o.ncomp == 4)
         set_quat_cell<T, NDIM, 4, FROM>(w, q, a.ncg, 4, b, u);
      else
         set_quat_cell<T, NDIM, 0, FROM>(w, q, a.ncg, o.ncomp, b, u);
      return;
   }
   const EllRowCoef<T> w = ell_row_coef<T, NDIM>(a, c, o, dinv);
   const T dudr = T(1) / w.diag;
   for (int m = 0; m < o.ncomp; m++) {
      QuatRowVals<T, NDIM> v;
      nbr_start<T, NDIM, FROM>(q, u + m * a.ncg, v);
      const T rv = b[m * a.ncg + q.c];
      const T res = FROM == 1 ? rv : ell_row_residual<T, NDIM>(w, dinv, rv, v);
      const T du = -res * dudr;
      u[m * a.ncg + q.c] = v.zc + du * T(1);
   }
}

// One colour of the red-black sweep of every slot on the colour-compact
// mapping: blockIdx.y is the slot, so the phase, orientation and composition
// blocks (and the components of each) of a level are one launch instead of one
// per block; on the small levels of a hierarchy or a V-cycle a launch costs
// 2-4 us whatever it computes.  FROM 1 and 2: the first red and black colours of
// a solve from zero, which read no solution values they know to be zero, so
// that nothing clears the solution first: 32 instead of 48 + 16 bytes a cell for
// the red colour of the FP32 orientation block.  The large levels are bound by
// HBM: at 256^3 with six FP32 components about 310 us a colour (80 bytes a
// cell, 4.3 TB/s; 390 us as separate launches with their ghost fills), the first
// red one 230 us.
template <typename T, int NDIM, bool SPLIT, bool WRAP, int FROM>
__global__ void __launch_bounds__(128) k_set_sweep(LevelArgs a, SweepSet<T> set, T di0, T di1,
                                                   T di2, T hi0, T hi1, T hi2,
                                                   const T* __restrict__ rhs, T* __restrict__ x,
                                                   int color)
{
   CellPos c;
   if (!cell_pos_color<NDIM>(a, 0, color, c)) return;
   const T dinv[3] = {di0, di1, di2}, hinv2[3] = {hi0, hi1, hi2};
   sweep_slot<T, NDIM, SPLIT, WRAP, FROM, -1, 0>(a, c, set.s[blockIdx.y], dinv, hinv2, rhs, x);
}

// The same of one block by itself (the smoother entry points, the block-by-block
// cycles of a hierarchy): its slot alone, of a known kind.  A set passes 1.4 kB
// of arguments whatever it holds and finds its slot when it runs: 3.8 us a launch
// on a level of some thousand cells, 3.1 us here.
template <typename T, int NDIM, int KIND, int QL>
__global__ void __launch_bounds__(128) k_block_sweep(LevelArgs a, SweepSlot<T> o, T di0, T di1,
                                                     T di2, T hi0, T hi1, T hi2,
                                                     const T* __restrict__ rhs,
                                                     T* __restrict__ x, int color)
{
   CellPos c;
   if (!cell_pos_color<NDIM>(a, 0, color, c)) return;
   const T dinv[3] = {di0, di1, di2}, hinv2[3] = {hi0, hi1, hi2};
   sweep_slot<T, NDIM, false, false, 0, KIND, QL>(a, c, o, dinv, hinv2, rhs, x);
}

// The residual of every slot, in one launch as k_set_sweep.
template <typename T, int NDIM, bool SPLIT>
__global__ void __launch_bounds__(256) k_set_residual(LevelArgs a, SweepSet<T> set, T di0, T di1,
                                                      T di2, T hi0, T hi1, T hi2,
                                                      const T* __restrict__ rhs,
                                                      const T* __restrict__ x,
                                                      T* __restrict__ res)
{
   CellPos c;
   if (!cell_pos(a, 0, c)) return;
   const SweepSlot<T>& o = set.s[blockIdx.y];
   const T* b = o.b ? o.b : rhs + o.comp * a.ncg;
   const T* u = x + o.comp * a.ncg;
   T* r = res + o.comp * a.ncg;
   const NbrIdx<NDIM> q = nbr_idx<NDIM, SPLIT, false>(a, c);
   if (o.kind == 1) {
      const T hinv2[3] = {hi0, hi1, hi2};
      const QuatRowCoef<T> w = quat_row_coef<T, NDIM>(a, c, o.D, o.sm, o.gamma, hinv2);
      for (int m = 0; m < o.ncomp; m++) {
         QuatRowVals<T, NDIM> v;
         nbr_start<T, NDIM, 0>(q, u + m * a.ncg, v);
         r[m * a.ncg + q.c] = b[m * a.ncg + q.c] - quat_row_apply<T, NDIM>(w, v);
      }
      return;
   }
   const T dinv[3] = {di0, di1, di2};
   const EllRowCoef<T> w = ell_row_coef<T, NDIM>(a, c, o, dinv);
   for (int m = 0; m < o.ncomp; m++) {
      QuatRowVals<T, NDIM> v;
      nbr_start<T, NDIM, 0>(q, u + m * a.ncg, v);
      r[m * a.ncg + q.c] = ell_row_residual<T, NDIM>(w, dinv, b[m * a.ncg + q.c], v);
   }
}

// Red residuals restricted, every slot in one launch.  After sweeps that end
// with the black colour the residual vanishes on black cells (a black update
// zeroes its own row's residual, and a black row couples its cell to red cells
// only), so the coarse right-hand side is the restriction of the red residuals:
// per coarse cell, its 2^(NDIM-1) red children's residuals in the
// restriction's summation order (each pair of x-children sums to its red
// member), without storing the fine residual.  Needs one checkerboard across
// patches and periodic ghosts (a zero-slope ghost would copy a black cell's
// new value into its own row); the host checks both.
template <typename T, int NDIM, int QL, bool SPLIT, bool WRAP>
__device__ __forceinline__ void set_resrestrict(const LevelArgs& ca, const LevelArgs& fa,
                                                const CellPos& p, const SweepSlot<T>& o,
                                                const T* dinv, const T* hinv2, const T* rhs,
                                                const T* x, T* bc, int m0)
{
   constexpr int N = QL > 0 ? QL : 1;
   const PatchDev fp = fa.P[ca.T[tile_index(ca)].patch];
   const T* b = (o.b ? o.b : rhs + o.comp * fa.ncg) + m0 * fa.ncg;
   const T* u = x + (o.comp + m0) * fa.ncg;
   T pr[N][4];
#pragma unroll
   for (int dz = 0; dz < (NDIM == 3 ? 2 : 1); dz++)
#pragma unroll
      for (int dy = 0; dy < 2; dy++) {
         CellPos c;
         c.pd = fp;
         c.j = 2 * p.j + dy;
         c.k = NDIM == 3 ? 2 * p.k + dz : 0;
         int gj = fp.lo[1] + c.j;
         int xs = (NDIM == 3) ? fp.lo[0] + gj + (fp.lo[2] + c.k) : fp.lo[1] + gj;
         int io = ((xs - (xs / 2) * 2) != 0) ? 1 : 0;  // red cells of the row (cell_pos_color)
         c.i = 2 * p.i + io;
         c.st[0] = 1;
         c.st[1] = fp.sy;
         c.st[2] = fp.sz;
         c.c0 = fp.cell_off + (c.i + fa.g) + (long long)(c.j + fa.g) * fp.sy +
                (long long)(c.k + fa.gz) * fp.sz;
         const NbrIdx<NDIM> q = nbr_idx<NDIM, SPLIT, WRAP>(fa, c);
         QuatRowVals<T, NDIM> v[N];
         T rv[N];
#pragma unroll
         for (int m = 0; m < N; m++) {
            nbr_start<T, NDIM, 0>(q, u + m * fa.ncg, v[m]);
            rv[m] = b[m * fa.ncg + q.c];
         }
         if (o.kind == 1) {
            const QuatRowCoef<T> w = quat_row_coef<T, NDIM>(fa, c, o.D, o.sm, o.gamma, hinv2);
#pragma unroll
            for (int m = 0; m < N; m++)
               pr[m][dy + 2 * dz] = rv[m] - quat_row_apply<T, NDIM>(w, v[m]);
         } else {
            const EllRowCoef<T> w = ell_row_coef<T, NDIM>(fa, c, o, dinv);
#pragma unroll
            for (int m = 0; m < N; m++)
               pr[m][dy + 2 * dz] = ell_row_residual<T, NDIM>(w, dinv, rv[m], v[m]);
         }
      }
   const long long co = (SPLIT ? split_at(ca, p, 0) : p.c0) + (o.comp + m0) * ca.ncg;
#pragma unroll
   for (int m = 0; m < N; m++) {
      T sum = pr[m][0] + pr[m][1];
      if (NDIM == 3) sum = sum + (pr[m][2] + pr[m][3]);
      bc[m * ca.ncg + co] = sum * (NDIM == 3 ? T(0.125) : T(0.25));
   }
}

template <typename T, int NDIM, bool SPLIT, bool WRAP>
__global__ void __launch_bounds__(256) k_set_resrestrict(LevelArgs ca, LevelArgs fa,
                                                         SweepSet<T> set, T di0, T di1, T di2,
                                                         T hi0, T hi1, T hi2,
                                                         const T* __restrict__ rhs,
                                                         const T* __restrict__ x,
                                                         T* __restrict__ bc)
{
   CellPos p;
   if (!cell_pos(ca, 0, p)) return;
   const SweepSlot<T>& o = set.s[blockIdx.y];
   const T dinv[3] = {di0, di1, di2}, hinv2[3] = {hi0, hi1, hi2};
   if (o.kind == 1 && o.ncomp == 4) {
      set_resrestrict<T, NDIM, 4, SPLIT, WRAP>(ca, fa, p, o, dinv, hinv2, rhs, x, bc, 0);
      return;
   }
   for (int m = 0; m < o.ncomp; m++)
      set_resrestrict<T, NDIM, 1, SPLIT, WRAP>(ca, fa, p, o, dinv, hinv2, rhs, x, bc, m);
}

// The same of one block by itself, of a known kind with QL components: the
// elliptic rows by themselves take 144 registers, with the orientation's in the same
// kernel 213.  192^3, FP64: elliptic block 46 us (60 as a set of one), orientation
// block of two components 157 us (196, one after the other).
template <typename T, int NDIM, int KIND, int QL>
__global__ void __launch_bounds__(256) k_block_resrestrict(LevelArgs ca, LevelArgs fa,
                                                           SweepSlot<T> o, T di0, T di1, T di2,
                                                           T hi0, T hi1, T hi2,
                                                           const T* __restrict__ rhs,
                                                           const T* __restrict__ x,
                                                           T* __restrict__ bc)
{
   CellPos p;
   if (!cell_pos(ca, 0, p)) return;
   const T dinv[3] = {di0, di1, di2}, hinv2[3] = {hi0, hi1, hi2};
   o.kind = KIND;
   set_resrestrict<T, NDIM, QL, false, false>(ca, fa, p, o, dinv, hinv2, rhs, x, bc, 0);
}

// ------------------------------------------------------------ launchers
static dim3 tblock() { return dim3(TX, TY); }
static dim3 cblock() { return dim3(TX / 2, TY); }

// Calls f(ndim, ql) with both as std::integral_constant: ql = ncomp for one,
// two or four components (all loads of a cell issued together), else 0.
template <class F>
static void quat_dispatch(int ndim, int ncomp, F&& f)
{
   using I2 = std::integral_constant<int, 2>;
   using I3 = std::integral_constant<int, 3>;
   auto by_ql = [&](auto nd) {
      switch (ncomp) {
      case 1: f(nd, std::integral_constant<int, 1>()); break;
      case 2: f(nd, std::integral_constant<int, 2>()); break;
      case 4: f(nd, std::integral_constant<int, 4>()); break;
      default: f(nd, std::integral_constant<int, 0>()); break;
      }
   };
   if (ndim == 3)
      by_ql(I3());
   else
      by_ql(I2());
}

// 1/h and 1/h^2 in the operator's precision, computed once per launch on the
// host (IEEE division: the device's value).
template <typename T>
static void recip(const double* dx, T* di)
{
   for (int d = 0; d < 3; d++) di[d] = T(1) / (T)dx[d];
}
template <typename T>
static void recip2(const double* dx, T* di)
{
   for (int d = 0; d < 3; d++) {
      T h = (T)dx[d];
      di[d] = T(1) / (h * h);
   }
}

int launch_phase_C(const Level& L, const ampe_model_params& p, double gamma,
                   const double* phi, const double* M, double* C, hipStream_t s)
{
   hipLaunchKernelGGL(k_phase_C, dim3(L.ncell_tiles), tblock(), 0, s, level_args(L), p, gamma,
                      phi, M, C);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

// Launch shape: column tiles (KZ planes per workgroup), or one-plane tiles
// when a per-tile reduction is requested (its callers reduce ncell_tiles
// partials).
static void shape(const Level& L, bool reduce, LevelArgs* a, int* grid)
{
   *a = reduce ? level_args(L) : level_args_col(L);
   *grid = reduce ? L.ncell_tiles : L.ncol_tiles;
}

template <typename T>
int sweep_add(SweepSet<T>& set, const SweepSlot<T>& proto, int comp, int ncomp)
{
   const int per = proto.kind == 1 ? ncomp : 4;
   for (int m = 0; m < ncomp; m += per) {
      if (set.n >= kMaxSlots) {
         set_error("sweep_add: too many preconditioner blocks");
         return -1;
      }
      SweepSlot<T>& o = set.s[set.n++];
      o = proto;
      o.comp = comp + m;
      o.ncomp = ncomp - m < per ? ncomp - m : per;
   }
   return 0;
}

// Calls f with the flags as std::integral_constant.
template <class F>
static void bool_dispatch(bool v, F&& f)
{
   if (v)
      f(std::true_type());
   else
      f(std::false_type());
}

template <typename T>
int launch_set_sweep(const Level& L, const SweepSet<T>& set, const double* dx, const T* rhs, T* x,
                     int color, const SetForm& form, hipStream_t s)
{
   T di[3], hi[3];
   recip(dx, di);
   recip2(dx, hi);
   dim3 g(L.ncell_tiles, set.n);
   const LevelArgs la = level_args(L);
   bool quat = false;
   for (int i = 0; i < set.n; i++) quat |= set.s[i].kind == 1;
   KernelTimer::Span span(quat ? KernelTimer::QUAT_RBGS : -1, s,
                          set_sweep_bytes(L, set, form.from));
   auto go = [&](auto nd, auto sp, auto wr, auto fr) {
      hipLaunchKernelGGL((k_set_sweep<T, decltype(nd)::value, decltype(sp)::value,
                                      decltype(wr)::value, decltype(fr)::value>),
                         g, cblock(), 0, s, la, set, di[0], di[1], di[2], hi[0], hi[1], hi[2],
                         rhs, x, color);
   };
   auto by_from = [&](auto nd, auto sp, auto wr) {
      if (form.from == 1)
         go(nd, sp, wr, std::integral_constant<int, 1>());
      else if (form.from == 2)
         go(nd, sp, wr, std::integral_constant<int, 2>());
      else
         go(nd, sp, wr, std::integral_constant<int, 0>());
   };
   const int rc = split_dispatch<T>(form.split, [&](auto sp) {
      bool_dispatch(form.wrap, [&](auto wr) {
         if (L.ndim == 3)
            by_from(std::integral_constant<int, 3>(), sp, wr);
         else
            by_from(std::integral_constant<int, 2>(), sp, wr);
      });
   });
   if (rc) return rc;
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_set_residual(const Level& L, const SweepSet<T>& set, const double* dx, const T* rhs,
                        const T* x, T* res, bool split, hipStream_t s)
{
   T di[3], hi[3];
   recip(dx, di);
   recip2(dx, hi);
   dim3 g(L.ncell_tiles, set.n);
   const LevelArgs la = level_args(L);
   auto go = [&](auto nd, auto sp) {
      hipLaunchKernelGGL((k_set_residual<T, decltype(nd)::value, decltype(sp)::value>), g,
                         tblock(), 0, s, la, set, di[0], di[1], di[2], hi[0], hi[1], hi[2], rhs, x,
                         res);
   };
   const int rc = split_dispatch<T>(split, [&](auto sp) {
      if (L.ndim == 3)
         go(std::integral_constant<int, 3>(), sp);
      else
         go(std::integral_constant<int, 2>(), sp);
   });
   if (rc) return rc;
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_set_resrestrict(const Level& coarse, const Level& fine, const SweepSet<T>& set,
                           const double* dx, const T* rhs, const T* x, T* b, const SetForm& form,
                           hipStream_t s)
{
   T di[3], hi[3];
   recip(dx, di);
   recip2(dx, hi);
   dim3 g(coarse.ncell_tiles, set.n);
   const LevelArgs ca = level_args(coarse), fa = level_args(fine);
   auto go = [&](auto nd, auto sp, auto wr) {
      hipLaunchKernelGGL((k_set_resrestrict<T, decltype(nd)::value, decltype(sp)::value,
                                            decltype(wr)::value>),
                         g, tblock(), 0, s, ca, fa, set, di[0], di[1], di[2], hi[0], hi[1], hi[2],
                         rhs, x, b);
   };
   const int rc = split_dispatch<T>(form.split, [&](auto sp) {
      bool_dispatch(form.wrap, [&](auto wr) {
         if (fine.ndim == 3)
            go(std::integral_constant<int, 3>(), sp, wr);
         else
            go(std::integral_constant<int, 2>(), sp, wr);
      });
   });
   if (rc) return rc;
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

// One block as a set of one slot (component 0 of the arrays passed).
template <typename T>
static SweepSet<T> ell_set(const EllOp<T>& op)
{
   SweepSet<T> set;
   set.n = 1;
   SweepSlot<T>& o = set.s[0];
   o.D = op.D;
   o.Dc = op.Dc;
   o.C = op.C;
   o.Cc = op.Cc;
   o.M = op.M;
   o.Mc = op.Mc;
   return set;
}
template <typename T>
static SweepSet<T> quat_set(const T* fc, const T* sm, double gamma, int ncomp)
{
   SweepSet<T> set;
   set.n = 1;
   SweepSlot<T>& o = set.s[0];
   o.kind = 1;
   o.ncomp = ncomp;
   o.D = fc;
   o.sm = sm;
   o.gamma = (T)gamma;
   return set;
}

template <typename T, class ND, class KIND, class QL>
static int block_sweep(ND, KIND, QL, const Level& L, const SweepSlot<T>& o, const double* dx,
                       const T* rhs, T* x, int color, hipStream_t s)
{
   T di[3], hi[3];
   recip(dx, di);
   recip2(dx, hi);
   hipLaunchKernelGGL((k_block_sweep<T, ND::value, KIND::value, QL::value>),
                      dim3(L.ncell_tiles), cblock(), 0, s, level_args(L), o, di[0], di[1], di[2],
                      hi[0], hi[1], hi[2], rhs, x, color);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_rbgs(const Level& L, const EllOp<T>& op, const double* dx, const T* rhs, T* u,
                int color, bool want_max, hipStream_t s)
{
   if (!want_max) {
      using I0 = std::integral_constant<int, 0>;
      const SweepSlot<T> o = ell_set(op).s[0];
      if (L.ndim == 3)
         return block_sweep<T>(std::integral_constant<int, 3>(), I0(), I0(), L, o, dx, rhs, u,
                               color, s);
      return block_sweep<T>(std::integral_constant<int, 2>(), I0(), I0(), L, o, dx, rhs, u, color,
                            s);
   }
   OpArgs<T> oa{op.D, op.Dc, op.C, op.Cc, op.M, op.Mc};
   double* part = L.partial;
   LevelArgs la = level_args(L);
   dim3 g(L.ncell_tiles);
   T di[3];
   recip(dx, di);
   if (L.ndim == 3)
      hipLaunchKernelGGL((k_rbgs<T, 3>), g, tblock(), 0, s, la, oa, di[0], di[1], di[2], rhs, u,
                         color, part);
   else
      hipLaunchKernelGGL((k_rbgs<T, 2>), g, tblock(), 0, s, la, oa, di[0], di[1], di[2], rhs, u,
                         color, part);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_residual(const Level& L, const EllOp<T>& op, const double* dx, const T* rhs,
                    const T* u, T* res, double* part, hipStream_t s)
{
   OpArgs<T> oa{op.D, op.Dc, op.C, op.Cc, op.M, op.Mc};
   LevelArgs la;
   int grid;
   shape(L, part != nullptr, &la, &grid);
   T di[3];
   recip(dx, di);
   if (L.ndim == 3)
      hipLaunchKernelGGL((k_residual<T, 3>), dim3(grid), tblock(), 0, s, la, oa, di[0], di[1],
                         di[2], rhs, u, res, part);
   else
      hipLaunchKernelGGL((k_residual<T, 2>), dim3(grid), tblock(), 0, s, la, oa, di[0], di[1],
                         di[2], rhs, u, res, part);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T, class ND, class KIND, class QL>
static int block_resrestrict(ND, KIND, QL, const Level& coarse, const Level& fine,
                             const SweepSlot<T>& o, const double* dx, const T* rhs, const T* x,
                             T* b, hipStream_t s)
{
   T di[3], hi[3];
   recip(dx, di);
   recip2(dx, hi);
   hipLaunchKernelGGL((k_block_resrestrict<T, ND::value, KIND::value, QL::value>),
                      dim3(coarse.ncell_tiles), tblock(), 0, s, level_args(coarse),
                      level_args(fine), o, di[0], di[1], di[2], hi[0], hi[1], hi[2], rhs, x, b);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_ell_resrestrict(const Level& coarse, const Level& fine, const EllOp<T>& op,
                           const double* dx, const T* rhs, const T* u, T* b, hipStream_t s)
{
   using I0 = std::integral_constant<int, 0>;
   using I1 = std::integral_constant<int, 1>;
   const SweepSlot<T> o = ell_set(op).s[0];
   if (fine.ndim == 3)
      return block_resrestrict<T>(std::integral_constant<int, 3>(), I0(), I1(), coarse, fine, o, dx,
                                  rhs, u, b, s);
   return block_resrestrict<T>(std::integral_constant<int, 2>(), I0(), I1(), coarse, fine, o, dx,
                               rhs, u, b, s);
}

template <typename T>
int launch_quat_rbgs(const Level& L, const T* fc, const T* sm, double gamma, const double* dx,
                     int ncomp, const T* rhs, T* z, int color, hipStream_t s)
{
   const SweepSet<T> set = quat_set(fc, sm, gamma, ncomp);
   KernelTimer::Span span(KernelTimer::QUAT_RBGS, s, set_sweep_bytes(L, set, 0));
   int rc = 0;
   quat_dispatch(L.ndim, ncomp, [&](auto nd, auto ql) {
      rc = block_sweep<T>(nd, std::integral_constant<int, 1>(), ql, L, set.s[0], dx, rhs, z, color,
                          s);
   });
   return rc;
}

template <typename T>
int launch_quat_rbgs_fused(const Level& L, const T* fc, const T* sm, double gamma,
                           const double* dx, int ncomp, const T* rhs, const T* zin, T* zout,
                           hipStream_t s)
{
   if (ncomp > 4) {
      set_error("launch_quat_rbgs_fused: at most four components");
      return -1;
   }
   T hi[3];
   recip2(dx, hi);
   LevelArgs la = level_args(L);
   dim3 g(L.ncell_tiles);
   {
      KernelTimer::Span span(KernelTimer::QUAT_RBGS, s, quat_rbgs_fused_bytes(L, ncomp, sizeof(T)));
      LevelArgs lm = level_args_march(L);
      dim3 gm(L.nmarch_tiles);
      if (L.ndim == 3)
         hipLaunchKernelGGL((k_quat_rbgs_fused<T, 3>), gm, tblock(), 0, s, lm, fc, sm, (T)gamma,
                            hi[0], hi[1], hi[2], ncomp, rhs, zin, zout);
      else
         hipLaunchKernelGGL((k_quat_rbgs_fused<T, 2>), gm, tblock(), 0, s, lm, fc, sm, (T)gamma,
                            hi[0], hi[1], hi[2], ncomp, rhs, zin, zout);
      AMPE_HIP_CHECK(hipGetLastError());
   }
   if (ghost_fill(L, zout, ncomp, s)) return -1;
   if (L.ndim == 3)
      hipLaunchKernelGGL((k_quat_rbgs_shell<T, 3>), g, tblock(), 0, s, la, fc, sm, (T)gamma,
                         hi[0], hi[1], hi[2], ncomp, rhs, zin, zout);
   else
      hipLaunchKernelGGL((k_quat_rbgs_shell<T, 2>), g, tblock(), 0, s, la, fc, sm, (T)gamma,
                         hi[0], hi[1], hi[2], ncomp, rhs, zin, zout);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_quat_residual(const Level& L, const T* fc, const T* sm, double gamma,
                         const double* dx, int ncomp, const T* rhs, const T* z, T* res,
                         double* part, hipStream_t s, bool split)
{
   LevelArgs la = level_args(L);
   dim3 g(L.ncell_tiles);
   T hi[3];
   recip2(dx, hi);
   const int rc = split_dispatch<T>(split, [&](auto sp) {
      quat_dispatch(L.ndim, ncomp, [&](auto ndim, auto ql) {
         hipLaunchKernelGGL((k_quat_residual<T, decltype(ndim)::value, decltype(ql)::value,
                                             decltype(sp)::value>),
                            g, tblock(), 0, s, la, fc, sm, (T)gamma, hi[0], hi[1], hi[2], ncomp,
                            rhs, z, res, part);
      });
   });
   if (rc) return rc;
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int launch_quat_resrestrict(const Level& coarse, const Level& fine, const T* fc, const T* sm,
                            double gamma, const double* dx, int ncomp, const T* rhs, const T* z,
                            T* b, hipStream_t s)
{
   if (ncomp != 1 && ncomp != 2 && ncomp != 4) {
      set_error("launch_quat_resrestrict: one, two or four components");
      return -1;
   }
   const SweepSet<T> set = quat_set(fc, sm, gamma, ncomp);
   int rc = 0;
   quat_dispatch(fine.ndim, ncomp, [&](auto nd, auto ql) {
      if constexpr (decltype(ql)::value > 0)
         rc = block_resrestrict<T>(nd, std::integral_constant<int, 1>(), ql, coarse, fine, set.s[0],
                                   dx, rhs, z, b, s);
   });
   return rc;
}

#define AMPE_INST(T)                                                                     \
   template int sweep_add<T>(SweepSet<T>&, const SweepSlot<T>&, int, int);               \
   template int launch_set_sweep<T>(const Level&, const SweepSet<T>&, const double*,     \
                                    const T*, T*, int, const SetForm&, hipStream_t);     \
   template int launch_set_residual<T>(const Level&, const SweepSet<T>&, const double*,  \
                                       const T*, const T*, T*, bool, hipStream_t);       \
   template int launch_set_resrestrict<T>(const Level&, const Level&, const SweepSet<T>&, \
                                          const double*, const T*, const T*, T*,         \
                                          const SetForm&, hipStream_t);                  \
   template int launch_rbgs<T>(const Level&, const EllOp<T>&, const double*, const T*, T*, \
                               int, bool, hipStream_t);                                  \
   template int launch_residual<T>(const Level&, const EllOp<T>&, const double*, const T*, \
                                   const T*, T*, double*, hipStream_t);                  \
   template int launch_quat_rbgs<T>(const Level&, const T*, const T*, double, const double*, \
                                    int, const T*, T*, int, hipStream_t);                \
   template int launch_quat_residual<T>(const Level&, const T*, const T*, double,         \
                                        const double*, int, const T*, const T*, T*,      \
                                        double*, hipStream_t, bool);
AMPE_INST(double)
AMPE_INST(float)
// by the entry points alone
template int launch_ell_resrestrict<double>(const Level&, const Level&, const EllOp<double>&,
                                            const double*, const double*, const double*, double*,
                                            hipStream_t);
template int launch_quat_resrestrict<double>(const Level&, const Level&, const double*,
                                             const double*, double, const double*, int,
                                             const double*, const double*, double*, hipStream_t);
template int launch_quat_rbgs_fused<double>(const Level&, const double*, const double*, double,
                                            const double*, int, const double*, const double*,
                                            double*, hipStream_t);

}  // namespace ampe
