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
// the dots waited for each other.  Modified Gram-Schmidt takes two basis vectors
// a pass (k_mgs).
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

// Sums of N runs of np values, ps apart, by the whole workgroup, the same in every
// one (fixed order).
template <int N>
__device__ __forceinline__ void sum_parts(const double* __restrict__ p, int np, int ps,
                                          double (&s)[N])
{
   if (np == 1) {
#pragma unroll
      for (int k = 0; k < N; k++) s[k] = p[k * ps];
      return;
   }
   __shared__ double sh[4][N];
   const int t = threadIdx.x + TX * threadIdx.y;
   double v[N];
#pragma unroll
   for (int k = 0; k < N; k++) v[k] = 0.0;
   for (int i = t; i < np; i += TX * TY)
#pragma unroll
      for (int k = 0; k < N; k++) v[k] += p[(long long)k * ps + i];
#pragma unroll
   for (int k = 0; k < N; k++) {
      for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o);
      if ((t & 63) == 0) sh[t >> 6][k] = v[k];
   }
   __syncthreads();
#pragma unroll
   for (int k = 0; k < N; k++) s[k] = (sh[0][k] + sh[1][k]) + (sh[2][k] + sh[3][k]);
}

// Two basis vectors and their normalisation factors.
struct VecPair {
   const double* v[2];
   double h[2];
};

// Modified Gram-Schmidt, two vectors a pass: z = src + c0 v0 + c1 v1 with
// c_k = -((s_k h_k) cv) h_k, s0 = src . v0 and s1 = (src + c0 v0) . v1 =
// src . v1 + c0 (v0 . v1), stored to dot[0] and dot[1].  parts: the np partial
// sums, ps apart, of src . v0, src . v1 and v0 . v1.  partial: the same sums of z and
// the next pair (NEXT 2), z . next (NEXT 1) or z . z (NEXT 0).  CUR 1: one vector;
// CUR 0: none, the first products (z is not written).
// Bound by memory.  One vector a pass reads z, ewt, the vector and the next one and
// writes z: five vectors' traffic for one; two a pass cost seven.  256^3, six
// components (805 MB a vector): 1114 us for two (5.1 TB/s), 742 us for one by
// itself; with the scaled basis (no ewt, one vector a pass) 596 us, and two
// passes more per iteration (1.3 ms).  An iteration at maxl = 30: 17.1 ms, 20.2 in the
// scaled form.
template <int CUR, int NEXT>
__global__ void __launch_bounds__(256) k_mgs(LevelArgs a, int nc, int ntiles, PrecOut src,
                                             VecPair cur, VecPair next, double cv,
                                             const double* __restrict__ parts, int np, int ps,
                                             double* __restrict__ dot,
                                             const double* __restrict__ ewt, double* z,
                                             double* __restrict__ partial)
{
   double co[2] = {0.0, 0.0};
   if (CUR > 0) {
      double s[CUR == 2 ? 3 : 1];
      sum_parts(parts, np, ps, s);
      co[0] = -((s[0] * cur.h[0]) * cv) * cur.h[0];
      if (CUR == 2) {
         s[1] = s[1] + co[0] * s[CUR == 2 ? 2 : 0];
         co[1] = -((s[1] * cur.h[1]) * cv) * cur.h[1];
      }
      if (blockIdx.x == 0 && threadIdx.x + threadIdx.y == 0)
         for (int k = 0; k < CUR; k++) dot[k] = s[k];
   }
   constexpr int NS = NEXT == 2 ? 3 : 1;
   CellPos c;
   double acc[NS];
#pragma unroll
   for (int k = 0; k < NS; k++) acc[k] = 0.0;
   if (cell_pos(a, 0, c)) {
      const double w = red_w(a, c.c0);
      const long long sp = src.sp0 < nc ? split_at(a, c, 0) : 0;
      const double sm = src.sm ? src.sm[c.c0] : 1.0;
      for (int m = 0; m < nc; m += 2) {
         const Pair p = pair_of(a, c, nc, m);
         double e[2], t[2], b[2][2], x[2][2];
#pragma unroll
         for (int j = 0; j < 2; j++) {
            e[j] = ewt[p.i[j]];
            t[j] = prec_out(a, src, c, sp, m + 1 < nc ? m + j : m, sm);
#pragma unroll
            for (int k = 0; k < CUR; k++) b[j][k] = cur.v[k][p.i[j]];
#pragma unroll
            for (int k = 0; k < NEXT; k++) x[j][k] = next.v[k][p.i[j]];
         }
#pragma unroll
         for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int k = 0; k < CUR; k++) t[j] = t[j] + co[k] * b[j][k];
            const double u = e[j] * t[j], wj = j ? w * p.on : w;
            if (NEXT == 0) {
               acc[0] += (u * u) * wj;
            } else {
               acc[0] += ((u * e[j]) * x[j][0]) * wj;
               if (NEXT == 2) {
                  acc[1] += ((u * e[j]) * x[j][1]) * wj;
                  acc[NS - 1] += (((e[j] * e[j]) * x[j][0]) * x[j][1]) * wj;
               }
            }
         }
         if (CUR > 0) {
            z[p.i[0]] = t[0];
            if (m + 1 < nc) z[p.i[1]] = t[1];
         }
      }
   }
   tile_store_sums(acc, NS, ntiles, partial);
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

// Up to this many tiles a pass sums the partial products of the pass before by
// itself, in every workgroup: at most twelve loads a thread; above, a reduction
// launch comes between (about 2 us and its gap).
constexpr int kSelfSumTiles = 1024;

int kry_mgs(const Level& L, int nc, const PrecOut& src, const VecList& vl, double cv,
            const double* ewt, double* z, double* sums, hipStream_t s)
{
   const int n = vl.n, nt = L.ncell_tiles;
   if (n < 1 || n > kMaxKrylov) {
      set_error("kry_mgs: too many vectors");
      return -1;
   }
   const bool self = nt <= kSelfSumTiles;
   // L.dred: the n products, and behind them the sums a pass starts from
   double* start = L.dred + kMaxKrylov;
   PrecOut from = src;
   VecPair cur{}, next{};
   // pass i takes vectors i - 2 and i - 1 out and forms the products of i and i + 1
   for (int i = 0; i < n + 2; i += 2) {
      const int take = i == 0 ? 0 : (i <= n ? 2 : 1), form = i >= n ? 0 : (i + 1 < n ? 2 : 1);
      cur = next;
      for (int k = 0; k < form; k++) {
         next.v[k] = vl.v[i + k];
         next.h[k] = vl.y[i + k];
      }
      const int half = (i >> 1) & 1;
      double* out = L.partial + 3LL * half * nt;
      const double* in = L.partial + 3LL * (1 - half) * nt;
      if (take && !self) {
         if (reduce_regions_dev(L, in, nt, take == 2 ? 3 : 1, start, s)) return -1;
         in = start;
      }
      const int np = self ? nt : 1, ps = self ? nt : 1;
      double* dot = L.dred + (i ? i - 2 : 0);
#define AMPE_MGS_CASE(CUR, NEXT)                                                             \
   if (take == CUR && form == NEXT)                                                          \
   AMPE_TILE_LAUNCH((k_mgs<CUR, NEXT>), nc, nt, from, cur, next, cv, in, np, ps, dot, ewt, z, out)
      AMPE_MGS_CASE(0, 1);
      AMPE_MGS_CASE(0, 2);
      AMPE_MGS_CASE(1, 0);
      AMPE_MGS_CASE(2, 0);
      AMPE_MGS_CASE(2, 1);
      AMPE_MGS_CASE(2, 2);
#undef AMPE_MGS_CASE
      if (take) {
         from = PrecOut{};
         from.z = z;
      }
      if (form == 0) return reduce_last(L, out, nt, n, sums, s);
   }
   return -1;
}

int kry_newton_update(const Level& L, int nc, const VecList& vl, const double* ewt, double* y,
                      double* sumsq, hipStream_t s)
{
   AMPE_TILE_LAUNCH(k_newton_update, nc, vl, ewt, y, L.partial);
   return reduce_partials(L, L.ncell_tiles, 1, 0, sumsq, s);
}

}  // namespace ampe
