// Fused vector kernels of the Newton-Krylov loop.  Each runs over the interior
// cells of a level (tile list) and all nc component blocks, performs the
// element-wise update of one or two steps of SPGMR / Newton in one pass and
// writes one partial sum per tile for the reduction that follows, so a
// Gram-Schmidt step costs one read of each operand instead of two or three.
// Ghost entries of Krylov vectors are not touched: every consumer that reads a
// stencil ghost-fills its input first.
//
// The error weights ewt stay out of the stored basis: z is a preconditioned
// vector as it is, SPGMR's scaled basis vector is ewt z hs with hs its
// normalisation.  The direction of a difference quotient is then z hs (no read of
// ewt, no division, and the increment, a constant of the normalised vector, needs
// no norm), the correction a plain sum, and the vector to orthogonalise is
// read where the preconditioner left it, in the dots and again in the update,
// and written once.  The coefficients go from the dots to the update on the
// device; the host reads them with the norm, once per iteration.
//
// All are bound by memory.  128^3, six components (100 MB a vector), time per
// call averaged over an integration (1 to 6 basis vectors), before with the
// scaled basis: dots 91 us (158), update 111 us (106; it reads ewt and the FP32 vector now,
// and no longer waits for the host), finish 78 us (97), mid
// 54 us (77).  Vectors are loaded two components at a time and for a compiled
// count of basis vectors (up to ten): behind a branch per vector the loads of
// the dots waited for each other.
#include "krylov.h"

namespace ampe {

__device__ __forceinline__ void tile_store_sum(double acc, double* __restrict__ partial)
{
   for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
   __shared__ double sh[4];
   int t = threadIdx.x + TX * threadIdx.y;
   if ((t & 63) == 0) sh[t >> 6] = acc;
   __syncthreads();
   if (t == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Per-tile sums of n values (n <= kMaxCgs) to partial[k * ntiles + tile].
template <int N>
__device__ __forceinline__ void tile_store_sums(const double (&acc)[N], int n, int ntiles,
                                                double* __restrict__ partial)
{
   __shared__ double sh[4][N];
   int t = threadIdx.x + TX * threadIdx.y;
#pragma unroll
   for (int k = 0; k < N; k++) {
      if (k >= n) break;
      double v = acc[k];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
      if ((t & 63) == 0) sh[t >> 6][k] = v;
   }
   __syncthreads();
   if (t < n) partial[(long long)t * ntiles + blockIdx.x] = (sh[0][t] + sh[1][t]) + (sh[2][t] + sh[3][t]);
}

// Components m and m + 1 of a cell; the second is the first again, with weight
// zero, when nc is odd.
struct Pair {
   long long i[2];
   double on;  // 1, or 0 for no second
};

__device__ __forceinline__ Pair pair_of(const LevelArgs& a, const CellPos& c, int nc, int m)
{
   Pair p;
   p.i[0] = m * a.ncg + c.c0;
   p.i[1] = m + 1 < nc ? p.i[0] + a.ncg : p.i[0];
   p.on = m + 1 < nc ? 1.0 : 0.0;
   return p;
}

// Component m of the vector src describes, at cell c.
__device__ __forceinline__ double prec_out(const LevelArgs& a, const PrecOut& src, const CellPos& c,
                                           long long sp, int m, double sm)
{
   const long long i = m * a.ncg;
   double v = src.u ? (double)src.u[i + (m >= src.sp0 ? sp : c.c0)] : src.z[i + c.c0];
   if (src.sm && in_range(m, src.iq, src.ql)) v = v * sm;
   return v;
}

// Workgroups from ntiles on take the ghosts (dst a copy of src), so that the
// stencils that follow need no launch of their own for them.
__global__ void __launch_bounds__(256) k_kry_mid(LevelArgs a, int nc, int ntiles, double sig,
                                                 const double* __restrict__ z, double h,
                                                 const double* __restrict__ ycur,
                                                 double* __restrict__ work2,
                                                 const long long* __restrict__ dst,
                                                 const long long* __restrict__ src, long long ng)
{
   long long from, to;
   if ((int)blockIdx.x < ntiles) {
      CellPos c;
      if (!cell_pos(a, 0, c)) return;
      from = to = c.c0;
   } else {
      const long long e = (long long)((int)blockIdx.x - ntiles) * (TX * TY) +
                          (int)(threadIdx.x + TX * threadIdx.y);
      if (e >= ng) return;
      to = dst[e];
      from = src[e];
   }
#pragma unroll 2
   for (int m = 0; m < nc; m++)
      work2[m * a.ncg + to] = sig * (z[m * a.ncg + from] * h) + ycur[m * a.ncg + from];
}

__global__ void __launch_bounds__(256) k_kry_finish(LevelArgs a, int nc, KryFin fin,
                                                    const double* __restrict__ jv)
{
   CellPos c;
   if (!cell_pos(a, 0, c)) return;
   const long long sp = fin.pin.sp0 < nc ? split_at(a, c, 0) : 0;
   const double sm = fin.pin.sm ? fin.pin.sm[c.c0] : 1.0;
   for (int m = 0; m < nc; m += 2) {
      const Pair p = pair_of(a, c, nc, m);
      double v[2];
#pragma unroll
      for (int e = 0; e < 2; e++) v[e] = kry_fin(fin, p.i[e], jv[p.i[e]]);
      prec_in(a, fin.pin, c, sp, m, v[0], sm, fin.out);
      if (m + 1 < nc) prec_in(a, fin.pin, c, sp, m + 1, v[1], sm, fin.out);
   }
}

__global__ void __launch_bounds__(256) k_newton_rhs(LevelArgs a, int nc, double gamma,
                                                    const double* __restrict__ f,
                                                    const double* __restrict__ y,
                                                    const double* __restrict__ ah, double* out,
                                                    PrecIn pin)
{
   CellPos c;
   if (!cell_pos(a, 0, c)) return;
   const long long sp = pin.sp0 < nc ? split_at(a, c, 0) : 0;
   const double sm = pin.sm ? pin.sm[c.c0] : 1.0;
   for (int m = 0; m < nc; m += 2) {
      const Pair p = pair_of(a, c, nc, m);
      double v[2];
#pragma unroll
      for (int e = 0; e < 2; e++) v[e] = gamma * f[p.i[e]] - (y[p.i[e]] - ah[p.i[e]]);
      prec_in(a, pin, c, sp, m, v[0], sm, out);
      if (m + 1 < nc) prec_in(a, pin, c, sp, m + 1, v[1], sm, out);
   }
}

// partial[k * ntiles + tile] = sum (ewt src)(ewt v[k]), k < n, then of (ewt src)^2.
// N: the count at compile time (-1: n at run time).
template <int N>
__global__ void __launch_bounds__(256) k_cgs_dots(LevelArgs a, int nc, int ntiles, PrecOut src,
                                                  VecList vl, const double* __restrict__ ewt,
                                                  double* __restrict__ partial)
{
   constexpr int NA = N >= 0 ? N : kMaxCgs - 1;
   const int n = N >= 0 ? N : vl.n;
   CellPos c;
   double acc[NA + 1];
#pragma unroll
   for (int k = 0; k <= NA; k++) acc[k] = 0.0;
   if (cell_pos(a, 0, c)) {
      const double w = red_w(a, c.c0);
      const long long sp = src.sp0 < nc ? split_at(a, c, 0) : 0;
      const double sm = src.sm ? src.sm[c.c0] : 1.0;
      for (int m = 0; m < nc; m += 2) {
         const Pair p = pair_of(a, c, nc, m);
         double e[2], t[2], z[2][NA];
#pragma unroll
         for (int j = 0; j < 2; j++) {
            e[j] = ewt[p.i[j]];
            t[j] = prec_out(a, src, c, sp, m + 1 < nc ? m + j : m, sm);
            if (N >= 0) {
#pragma unroll
               for (int k = 0; k < NA; k++) z[j][k] = vl.v[k][p.i[j]];
            }
         }
#pragma unroll
         for (int j = 0; j < 2; j++) {
            const double v = e[j] * t[j], wj = j ? w * p.on : w, u = (v * e[j]) * wj;
            if (N >= 0) {
#pragma unroll
               for (int k = 0; k < NA; k++) acc[k] += u * z[j][k];
               acc[NA] += (v * v) * wj;
            } else {
#pragma unroll
               for (int k = 0; k <= NA; k++) {
                  if (k < n) acc[k] += u * vl.v[k][p.i[j]];
                  if (k == n) acc[k] += (v * v) * wj;
               }
            }
         }
      }
   }
   tile_store_sums(acc, n + 1, ntiles, partial);
}

// z = src + sum_k c_k v[k], c_k = -((sums[k] vl.y[k]) cv) vl.y[k];
// partial = sum (ewt z)^2
template <int N>
__global__ void __launch_bounds__(256) k_cgs_update(LevelArgs a, int nc, PrecOut src, VecList vl,
                                                    double cv, const double* __restrict__ sums,
                                                    const double* __restrict__ ewt, double* z,
                                                    double* __restrict__ partial)
{
   constexpr int NA = N >= 0 ? N : kMaxCgs - 1;
   const int n = N >= 0 ? N : vl.n;
   CellPos c;
   double acc = 0.0;
   if (cell_pos(a, 0, c)) {
      const double w = red_w(a, c.c0);
      const long long sp = src.sp0 < nc ? split_at(a, c, 0) : 0;
      const double sm = src.sm ? src.sm[c.c0] : 1.0;
      double co[NA + 1];
#pragma unroll
      for (int k = 0; k < NA; k++)
         if (k < n) co[k] = -((sums[k] * vl.y[k]) * cv) * vl.y[k];
      for (int m = 0; m < nc; m += 2) {
         const Pair p = pair_of(a, c, nc, m);
         double e[2], t[2], b[2][NA + 1];
#pragma unroll
         for (int j = 0; j < 2; j++) {
            e[j] = ewt[p.i[j]];
            t[j] = prec_out(a, src, c, sp, m + 1 < nc ? m + j : m, sm);
            if (N >= 0) {
#pragma unroll
               for (int k = 0; k < NA; k++) b[j][k] = vl.v[k][p.i[j]];
            }
         }
#pragma unroll
         for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int k = 0; k < NA; k++)
               if (k < n) t[j] = t[j] + co[k] * (N >= 0 ? b[j][k] : vl.v[k][p.i[j]]);
            const double v = e[j] * t[j];
            acc += (v * v) * (j ? w * p.on : w);
         }
         z[p.i[0]] = t[0];
         if (m + 1 < nc) z[p.i[1]] = t[1];
      }
   }
   tile_store_sum(acc, partial);
}

// Sum of np values by the whole workgroup, the same in every one (fixed order).
__device__ __forceinline__ double sum_parts(const double* __restrict__ p, int np)
{
   if (np == 1) return p[0];
   __shared__ double sh[4];
   const int t = threadIdx.x + TX * threadIdx.y;
   double v = 0.0;
   for (int i = t; i < np; i += TX * TY) v += p[i];
   for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
   if ((t & 63) == 0) sh[t >> 6] = v;
   __syncthreads();
   return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// One step of modified Gram-Schmidt and the product of the next:
// z = src + c v, c = -((s hv) cv) hv with s the sum of the np values at parts
// (stored to *dot); partial = sum (ewt z)(ewt next), or (ewt z)^2 (next null).
// v null: no update (z is not written), the first product.
__global__ void __launch_bounds__(256) k_mgs(LevelArgs a, int nc, PrecOut src,
                                             const double* __restrict__ v, double hv, double cv,
                                             const double* __restrict__ parts, int np, double* dot,
                                             const double* __restrict__ next,
                                             const double* __restrict__ ewt, double* z,
                                             double* __restrict__ partial)
{
   double co = 0.0;
   if (v) {
      const double s = sum_parts(parts, np);
      if (np > 1 && blockIdx.x == 0 && threadIdx.x + threadIdx.y == 0) *dot = s;
      co = -((s * hv) * cv) * hv;
   }
   CellPos c;
   double acc = 0.0;
   if (cell_pos(a, 0, c)) {
      const double w = red_w(a, c.c0);
      const long long sp = src.sp0 < nc ? split_at(a, c, 0) : 0;
      const double sm = src.sm ? src.sm[c.c0] : 1.0;
      for (int m = 0; m < nc; m += 2) {
         const Pair p = pair_of(a, c, nc, m);
         double e[2], t[2], b[2], x[2];
#pragma unroll
         for (int j = 0; j < 2; j++) {
            e[j] = ewt[p.i[j]];
            t[j] = prec_out(a, src, c, sp, m + 1 < nc ? m + j : m, sm);
            b[j] = v ? v[p.i[j]] : 0.0;
            x[j] = next ? next[p.i[j]] : 0.0;
         }
#pragma unroll
         for (int j = 0; j < 2; j++) {
            if (v) t[j] = t[j] + co * b[j];
            const double u = e[j] * t[j];
            acc += (next ? (u * e[j]) * x[j] : u * u) * (j ? w * p.on : w);
         }
         if (v) {
            z[p.i[0]] = t[0];
            if (m + 1 < nc) z[p.i[1]] = t[1];
         }
      }
   }
   tile_store_sum(acc, partial);
}

__global__ void __launch_bounds__(256) k_newton_update(LevelArgs a, int nc, VecList vl,
                                                       const double* __restrict__ ewt,
                                                       double* __restrict__ y,
                                                       double* __restrict__ partial)
{
   CellPos c;
   double acc = 0.0;
   if (cell_pos(a, 0, c)) {
      const double w = red_w(a, c.c0);
      for (int m = 0; m < nc; m += 2) {
         const Pair p = pair_of(a, c, nc, m);
         double x[2] = {0.0, 0.0}, e[2], yo[2];
#pragma unroll
         for (int j = 0; j < 2; j++) {
            e[j] = ewt[p.i[j]];
            yo[j] = y[p.i[j]];
         }
         for (int k = 0; k < vl.n; k++) {
            const double* __restrict__ v = vl.v[k];
            const double b0 = v[p.i[0]], b1 = v[p.i[1]];
            x[0] = x[0] + vl.y[k] * b0;
            x[1] = x[1] + vl.y[k] * b1;
         }
#pragma unroll
         for (int j = 0; j < 2; j++) {
            const double t = x[j] * e[j];
            acc += (t * t) * (j ? w * p.on : w);
         }
         y[p.i[0]] = yo[0] + x[0];
         if (m + 1 < nc) y[p.i[1]] = yo[1] + x[1];
      }
   }
   tile_store_sum(acc, partial);
}

#define AMPE_TILE_LAUNCH(KER, ...)                                                        \
   do {                                                                                   \
      hipLaunchKernelGGL(KER, dim3(L.ncell_tiles), dim3(TX, TY), 0, s, level_args(L),      \
                         __VA_ARGS__);                                                    \
      AMPE_HIP_CHECK(hipGetLastError());                                                  \
   } while (0)

int kry_mid(const Level& L, int nc, double sig, const double* z, double h, const double* ycur,
            double* work2, bool ghosts, hipStream_t s)
{
   const long long ng = ghosts ? L.nghost : 0;
   hipLaunchKernelGGL(k_kry_mid, dim3(L.ncell_tiles + (unsigned)((ng + TX * TY - 1) / (TX * TY))),
                      dim3(TX, TY), 0, s, level_args(L), nc, L.ncell_tiles, sig, z, h, ycur, work2,
                      L.ghost_dst, L.ghost_src, ng);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

int kry_finish(const Level& L, int nc, const KryFin& fin, const double* jv, hipStream_t s)
{
   AMPE_TILE_LAUNCH(k_kry_finish, nc, fin, jv);
   return 0;
}

int kry_newton_rhs(const Level& L, int nc, double gamma, const double* f, const double* y,
                   const double* ah, double* out, const PrecIn& pin, hipStream_t s)
{
   AMPE_TILE_LAUNCH(k_newton_rhs, nc, gamma, f, y, ah, out, pin);
   return 0;
}

static int cgs_dots(const Level& L, int nc, const PrecOut& src, const VecList& vl,
                    const double* ewt, hipStream_t s)
{
#define AMPE_CGS_CASE(N)                                                                    \
   case N:                                                                                  \
      AMPE_TILE_LAUNCH(k_cgs_dots<N>, nc, L.ncell_tiles, src, vl, ewt, L.partial);           \
      return 0;
   switch (vl.n) {
      AMPE_CGS_CASE(1) AMPE_CGS_CASE(2) AMPE_CGS_CASE(3) AMPE_CGS_CASE(4) AMPE_CGS_CASE(5)
      AMPE_CGS_CASE(6) AMPE_CGS_CASE(7) AMPE_CGS_CASE(8) AMPE_CGS_CASE(9) AMPE_CGS_CASE(10)
   }
#undef AMPE_CGS_CASE
   AMPE_TILE_LAUNCH(k_cgs_dots<-1>, nc, L.ncell_tiles, src, vl, ewt, L.partial);
   return 0;
}

static int cgs_update(const Level& L, int nc, const PrecOut& src, const VecList& vl, double cv,
                      const double* ewt, double* z, hipStream_t s)
{
#define AMPE_CGS_CASE(N)                                                                    \
   case N:                                                                                  \
      AMPE_TILE_LAUNCH(k_cgs_update<N>, nc, src, vl, cv, L.dred, ewt, z, L.partial);         \
      return 0;
   switch (vl.n) {
      AMPE_CGS_CASE(0) AMPE_CGS_CASE(1) AMPE_CGS_CASE(2) AMPE_CGS_CASE(3) AMPE_CGS_CASE(4)
      AMPE_CGS_CASE(5) AMPE_CGS_CASE(6) AMPE_CGS_CASE(7) AMPE_CGS_CASE(8) AMPE_CGS_CASE(9)
      AMPE_CGS_CASE(10)
   }
#undef AMPE_CGS_CASE
   AMPE_TILE_LAUNCH(k_cgs_update<-1>, nc, src, vl, cv, L.dred, ewt, z, L.partial);
   return 0;
}

int kry_start(const Level& L, int nc, const PrecOut& src, const double* ewt, double* z,
              double* sumsq, hipStream_t s)
{
   VecList vl;
   vl.n = 0;
   if (cgs_update(L, nc, src, vl, 0.0, ewt, z, s)) return -1;
   return reduce_partials(L, L.ncell_tiles, 1, 0, sumsq, s);
}

int kry_cgs(const Level& L, int nc, const PrecOut& src, const VecList& vl, double cv,
            const double* ewt, double* z, double* sums, hipStream_t s)
{
   const int n = vl.n;
   if (n < 1 || n + 1 > kMaxCgs) {
      set_error("kry_cgs: too many vectors");
      return -1;
   }
   if (cgs_dots(L, nc, src, vl, ewt, s)) return -1;
   if (reduce_regions_dev(L, L.partial, L.ncell_tiles, n + 1, L.dred, s)) return -1;
   if (cgs_update(L, nc, src, vl, cv, ewt, z, s)) return -1;
   double h[kMaxCgs + 1];
   if (reduce_last(L, L.partial, L.ncell_tiles, n + 1, h, s)) return -1;
   for (int k = 0; k < n; k++) sums[k] = h[k];
   sums[n + 1] = h[n];
   sums[n] = h[n + 1];
   return 0;
}

// Up to this many tiles a step sums the partial products of the step before by
// itself, in every workgroup: four loads a thread (128^2 has 64 tiles: 5.1 us a
// step); above, a reduction launch comes between (about 2 us and its gap).
constexpr int kSelfSumTiles = 1024;

int kry_mgs(const Level& L, int nc, const PrecOut& src, const VecList& vl, double cv,
            const double* ewt, double* z, double* sums, hipStream_t s)
{
   const int n = vl.n, nt = L.ncell_tiles;
   if (n < 1 || n > kMaxKrylov) {
      set_error("kry_mgs: too many vectors");
      return -1;
   }
   const bool self = nt > 1 && nt <= kSelfSumTiles;
   PrecOut in;
   in.z = z;
   AMPE_TILE_LAUNCH(k_mgs, nc, src, nullptr, 0.0, 0.0, nullptr, 0, nullptr, vl.v[0], ewt, nullptr,
                    L.partial);
   for (int i = 0; i < n; i++) {
      double* from = L.partial + (long long)(i & 1) * nt;
      double* to = L.partial + (long long)((i + 1) & 1) * nt;
      if (!self && reduce_regions_dev(L, from, nt, 1, L.dred + i, s)) return -1;
      AMPE_TILE_LAUNCH(k_mgs, nc, i ? in : src, vl.v[i], vl.y[i], cv, self ? from : L.dred + i,
                       self ? nt : 1, L.dred + i, i + 1 < n ? vl.v[i + 1] : nullptr, ewt, z, to);
   }
   return reduce_last(L, L.partial + (long long)(n & 1) * nt, nt, n, sums, s);
}

int kry_newton_update(const Level& L, int nc, const VecList& vl, const double* ewt, double* y,
                      double* sumsq, hipStream_t s)
{
   AMPE_TILE_LAUNCH(k_newton_update, nc, vl, ewt, y, L.partial);
   return reduce_partials(L, L.ncell_tiles, 1, 0, sumsq, s);
}

}  // namespace ampe
