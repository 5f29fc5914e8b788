// Geometric multigrid below one patch level (see mg.h).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "mg.h"

namespace ampe {

// ------------------------------------------------------------ transfers
// Coarse cell = mean of its 2^NDIM children (fixed summation order).
// SPLIT: f and c in the row parity-split layout (the two children of a row
// sit at the split positions of their columns; rows and planes as natural).
template <typename T, int NDIM, bool SPLIT>
__global__ void __launch_bounds__(256) k_restrict_cell(LevelArgs ca, LevelArgs fa, int ncomp,
                                                       const T* __restrict__ f,
                                                       T* __restrict__ c)
{
   CellPos p;
   if (!cell_pos(ca, 0, p)) return;
   const PatchDev fp = fa.P[ca.T[tile_index(ca)].patch];
   int fk = NDIM == 3 ? 2 * p.k : 0;
   const int ig = 2 * p.i + fa.g;
   const long long row = fp.cell_off + (long long)(2 * p.j + fa.g) * fp.sy +
                         (long long)(fk + fa.gz) * fp.sz;
   const long long f0 = SPLIT ? row + split_col(ig, fp.sy) : row + ig;
   const long long f1 = SPLIT ? row + split_col(ig + 1, fp.sy) : row + ig + 1;
   const long long co = SPLIT ? split_at(ca, p, 0) : p.c0;
   const long long sy = fp.sy, sz = fp.sz;
   for (int m = 0; m < ncomp; m++) {
      const T* fm = f + m * fa.ncg;
      T s = (fm[f0] + fm[f1]) + (fm[f0 + sy] + fm[f1 + sy]);
      if (NDIM == 3) s = s + ((fm[f0 + sz] + fm[f1 + sz]) + (fm[f0 + sz + sy] + fm[f1 + sz + sy]));
      c[m * ca.ncg + co] = s * (NDIM == 3 ? T(0.125) : T(0.25));
   }
}

// Coarse face = mean of the fine faces covering it.
template <typename T, int NDIM>
__global__ void __launch_bounds__(256) k_restrict_side(LevelArgs ca, LevelArgs fa,
                                                       const T* __restrict__ f,
                                                       T* __restrict__ c)
{
   CellPos p;
   if (!cell_pos(ca, 1, p)) return;
   if (NDIM == 2 && p.k > 0) return;
   const PatchDev fp = fa.P[ca.T[tile_index(ca)].patch];
   for (int d = 0; d < NDIM; d++) {
      bool ok = (p.i < p.pd.nx + (d == 0)) && (p.j < p.pd.ny + (d == 1)) &&
                (NDIM == 2 || p.k < p.pd.nz + (d == 2));
      if (!ok) continue;
      int b[3] = {2 * p.i, 2 * p.j, NDIM == 3 ? 2 * p.k : 0};
      int t1 = (d == 0) ? 1 : 0;  // first transverse direction
      int t2 = (d == 2) ? 1 : 2;  // second transverse direction (3-D)
      T s = 0;
      for (int a = 0; a < 2; a++)
         for (int e = 0; e < (NDIM == 3 ? 2 : 1); e++) {
            int q[3] = {b[0], b[1], b[2]};
            q[t1] += a;
            if (NDIM == 3) q[t2] += e;
            T v = f[face_idx(fa, fp, d, q[0], q[1], q[2])];
            s = (a == 0 && e == 0) ? v : s + v;
         }
      c[face_idx(ca, p.pd, d, p.i, p.j, p.k)] = s * (NDIM == 3 ? T(0.25) : T(0.5));
   }
}

// Fine cell += coarse correction: ORDER 1 tri/bilinear interpolation (weights
// 3/4 toward the parent, 1/4 toward the coarse neighbour on the cell's side in
// each direction; the coarse field needs filled ghosts unless WRAP, the one
// patch of a periodic level, whose neighbours across the boundary are read at
// its other side), ORDER 0 the parent value (constant refinement).  A
// workgroup takes the components blockIdx.y, blockIdx.y + gridDim.y, ...
template <typename T, int NDIM, int ORDER>
__device__ __forceinline__ T prolong_value(const T* __restrict__ x, long long c0, long long c1,
                                           long long oj, long long ok)
{
   if (ORDER == 0) return x[c0];
   if (NDIM == 2)
      return T(9.0 / 16.0) * x[c0] + T(3.0 / 16.0) * (x[c1] + x[c0 + oj]) +
             T(1.0 / 16.0) * x[c1 + oj];
   return T(27.0 / 64.0) * x[c0] + T(9.0 / 64.0) * ((x[c1] + x[c0 + oj]) + x[c0 + ok]) +
          T(3.0 / 64.0) * ((x[c1 + oj] + x[c1 + ok]) + x[c0 + oj + ok]) +
          T(1.0 / 64.0) * x[c1 + oj + ok];
}

// Offset from coarse position i of n along a stride st to its neighbour on the
// low (hi = 0) or high side.
template <bool WRAP>
__device__ __forceinline__ long long nbr_off(int i, int n, long long st, int hi)
{
   if (hi) return (WRAP && i == n - 1) ? -(long long)(n - 1) * st : st;
   return (WRAP && i == 0) ? (long long)(n - 1) * st : -st;
}

template <typename T, int NDIM, int ORDER, bool WRAP>
__global__ void __launch_bounds__(256) k_prolong_add(LevelArgs fa, LevelArgs ca, int ncomp,
                                                     const T* __restrict__ xc,
                                                     T* __restrict__ xf)
{
   CellPos p;
   if (!cell_pos(fa, 0, p)) return;
   const PatchDev cp = ca.P[fa.T[tile_index(fa)].patch];
   const int I = p.i >> 1, J = p.j >> 1, K = NDIM == 3 ? (p.k >> 1) : 0;
   const long long c0 = cp.cell_off + (I + ca.g) + (long long)(J + ca.g) * cp.sy +
                        (long long)(K + ca.gz) * cp.sz;
   const long long c1 = c0 + nbr_off<WRAP>(I, cp.nx, 1, p.i & 1);
   const long long oj = nbr_off<WRAP>(J, cp.ny, cp.sy, p.j & 1);
   const long long ok = NDIM == 3 ? nbr_off<WRAP>(K, cp.nz, cp.sz, p.k & 1) : 0;
   for (int m = blockIdx.y; m < ncomp; m += gridDim.y) {
      const T v = prolong_value<T, NDIM, ORDER>(xc + m * ca.ncg, c0, c1, oj, ok);
      T* y = xf + m * fa.ncg;
      y[p.c0] = y[p.c0] + v;
   }
}

// The split-layout interpolation per coarse cell: a thread adds the
// correction to the 2^NDIM children of its coarse cell (consecutive lanes:
// consecutive coarse cells, so for each child offset the fine updates are
// contiguous in the split layout), each child's value by the formula and
// summation order of the natural form.
template <typename T, int NDIM, bool WRAP>
__global__ void __launch_bounds__(256) k_prolong_add_cc(LevelArgs fa, LevelArgs ca,
                                                        const T* __restrict__ xc,
                                                        T* __restrict__ xf)
{
   CellPos p;
   if (!cell_pos(ca, 0, p)) return;
   const PatchDev fp = fa.P[ca.T[tile_index(ca)].patch];
   const int sy = p.pd.sy, nx = p.pd.nx;
   const int ig = p.i + ca.g;
   const long long row = p.c0 - ig;
   const long long c0 = row + split_col(ig, sy);
   const long long cm = row + split_col(ig + (int)nbr_off<WRAP>(p.i, nx, 1, 0), sy);
   const long long cp = row + split_col(ig + (int)nbr_off<WRAP>(p.i, nx, 1, 1), sy);
   const T* x = xc + blockIdx.y * ca.ncg;
   T* y = xf + blockIdx.y * fa.ncg;
   // every child's old value before the first update: the compiler cannot see
   // that the children differ, and would wait for each store
   long long fo[8];
   T old[8];
#pragma unroll
   for (int e = 0; e < (NDIM == 3 ? 8 : 4); e++) {
      const int fi = 2 * p.i + (e & 1), fj = 2 * p.j + ((e >> 1) & 1);
      const int fk = NDIM == 3 ? 2 * p.k + (e >> 2) : 0;
      fo[e] = fp.cell_off + split_col(fi + fa.g, fp.sy) + (long long)(fj + fa.g) * fp.sy +
              (long long)(fk + fa.gz) * fp.sz;
      old[e] = y[fo[e]];
   }
#pragma unroll
   for (int e = 0; e < (NDIM == 3 ? 8 : 4); e++) {
      const long long oj = nbr_off<WRAP>(p.j, p.pd.ny, sy, (e >> 1) & 1);
      const long long ok = NDIM == 3 ? nbr_off<WRAP>(p.k, p.pd.nz, p.pd.sz, e >> 2) : 0;
      y[fo[e]] = old[e] + prolong_value<T, NDIM, 1>(x, c0, (e & 1) ? cp : cm, oj, ok);
   }
}

template <typename T>
int mg_restrict_cell(const Level& coarse, const Level& fine, int ncomp, const T* f, T* c,
                     hipStream_t s, bool split)
{
   dim3 g(coarse.ncell_tiles), b(TX, TY);
   LevelArgs ca = level_args(coarse), fa = level_args(fine);
   auto go = [&](auto nd, auto sp) {
      hipLaunchKernelGGL((k_restrict_cell<T, decltype(nd)::value, decltype(sp)::value>), g, b, 0,
                         s, ca, fa, ncomp, f, c);
   };
   const int rc = split_dispatch<T>(split, [&](auto sp) {
      if (coarse.ndim == 3)
         go(std::integral_constant<int, 3>(), sp);
      else
         go(std::integral_constant<int, 2>(), sp);
   });
   if (rc) return rc;
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int mg_restrict_side(const Level& coarse, const Level& fine, const T* f, T* c, hipStream_t s)
{
   if (coarse.ndim == 3)
      hipLaunchKernelGGL((k_restrict_side<T, 3>), dim3(coarse.nface_tiles), dim3(TX, TY), 0, s,
                         level_args(coarse, true), level_args(fine), f, c);
   else
      hipLaunchKernelGGL((k_restrict_side<T, 2>), dim3(coarse.nface_tiles), dim3(TX, TY), 0, s,
                         level_args(coarse, true), level_args(fine), f, c);
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

template <typename T>
int mg_prolong_add(const Level& fine, const Level& coarse, int ncomp, int order, const T* xc,
                   T* xf, hipStream_t s, bool split, bool wrap)
{
   if (ncomp <= 0) return 0;
   // constant refinement: the components one after the other, the parent's place
   // found once (192^3, four components: 81 us, 95 with a workgroup each);
   // interpolated, where each component loads eight values, a workgroup each
   // (1024 x 768: 25.5 us, 26.5 one after the other; 192^3 141 us either way)
   dim3 gf(fine.ncell_tiles, order == 0 ? 1 : ncomp);
   dim3 gc(coarse.ncell_tiles, ncomp), b(TX, TY);
   LevelArgs fa = level_args(fine), ca = level_args(coarse);
   if (split && order == 0) {
      set_error("mg_prolong_add: the split layout has the interpolated form only");
      return -1;
   }
   auto go = [&](auto nd, auto sp, auto wr) {
      constexpr int ND = decltype(nd)::value;
      constexpr bool WR = decltype(wr)::value;
      if constexpr (decltype(sp)::value)
         hipLaunchKernelGGL((k_prolong_add_cc<T, ND, WR>), gc, b, 0, s, fa, ca, xc, xf);
      else if (order == 0)
         hipLaunchKernelGGL((k_prolong_add<T, ND, 0, false>), gf, b, 0, s, fa, ca, ncomp, xc, xf);
      else
         hipLaunchKernelGGL((k_prolong_add<T, ND, 1, WR>), gf, b, 0, s, fa, ca, ncomp, xc, xf);
   };
   const int rc = split_dispatch<T>(split, [&](auto sp) {
      auto by_wrap = [&](auto nd) {
         if (wrap)
            go(nd, sp, std::true_type());
         else
            go(nd, sp, std::false_type());
      };
      if (fine.ndim == 3)
         by_wrap(std::integral_constant<int, 3>());
      else
         by_wrap(std::integral_constant<int, 2>());
   });
   if (rc) return rc;
   AMPE_HIP_CHECK(hipGetLastError());
   return 0;
}

bool is_coarsening(const Level& coarse, const Level& fine)
{
   if (coarse.ndim != fine.ndim || coarse.npatch != fine.npatch) return false;
   for (int p = 0; p < fine.npatch; p++) {
      const PatchDev& f = fine.hp[p];
      const PatchDev& c = coarse.hp[p];
      int nf[3] = {f.nx, f.ny, f.nz}, nc[3] = {c.nx, c.ny, c.nz};
      for (int a = 0; a < fine.ndim; a++)
         if ((f.lo[a] & 1) || (nf[a] & 1) || c.lo[a] * 2 != f.lo[a] || nc[a] * 2 != nf[a])
            return false;
   }
   return true;
}

// ------------------------------------------------------------ hierarchy
static bool halvable(const Level& L, int min_cells)
{
   int nd = L.ndim;
   for (const PatchDev& d : L.hp) {
      int n[3] = {d.nx, d.ny, d.nz};
      for (int a = 0; a < nd; a++) {
         if ((d.lo[a] & 1) || (n[a] & 1) || n[a] / 2 < min_cells) return false;
      }
   }
   if (L.periodic)
      for (int a = 0; a < nd; a++) {
         int ext = L.pbox.hi[a] - L.pbox.lo[a] + 1;
         if ((L.pbox.lo[a] & 1) || (ext & 1)) return false;
      }
   return true;
}

template <typename T>
static int talloc(T** p, size_t n)
{
   if (hipMalloc(p, sizeof(T) * std::max<size_t>(n, 1)) != hipSuccess) return -1;
   return hipMemset(*p, 0, sizeof(T) * std::max<size_t>(n, 1)) == hipSuccess ? 0 : -1;
}

template <typename T>
int mg_create(const Level& fine, const double* dx, int ncomp_max, int max_levels, int min_cells,
              Mg<T>** out)
{
   Mg<T>* m = new Mg<T>();
   m->ncomp_max = ncomp_max;
   MgLevel<T> l0;
   l0.L = const_cast<Level*>(&fine);
   for (int a = 0; a < 3; a++) l0.dx[a] = dx[a];
   int rc = talloc(&l0.r, checker_ok(fine) ? 1 : (size_t)ncomp_max * fine.ncg);
   m->lv.push_back(l0);
   if (max_levels < 1) max_levels = 1;
   while (!rc && (int)m->lv.size() < max_levels && halvable(*m->lv.back().L, min_cells)) {
      const Level& F = *m->lv.back().L;
      std::vector<ampe_box> boxes(F.npatch);
      for (int p = 0; p < F.npatch; p++) {
         const PatchDev& d = F.hp[p];
         int n[3] = {d.nx, d.ny, d.nz};
         for (int a = 0; a < 3; a++) {
            boxes[p].lo[a] = a < F.ndim ? d.lo[a] / 2 : 0;
            boxes[p].hi[a] = a < F.ndim ? d.lo[a] / 2 + n[a] / 2 - 1 : 0;
         }
      }
      ampe_box pb;
      for (int a = 0; a < 3; a++) {
         pb.lo[a] = F.pbox.lo[a] / 2;
         pb.hi[a] = (F.pbox.hi[a] + 1) / 2 - 1;
      }
      MgLevel<T> c;
      if (level_create(F.ndim, boxes.data(), F.npatch, F.g, F.periodic ? &pb : nullptr, &c.L)) {
         rc = -1;
         break;
      }
      for (int a = 0; a < 3; a++) c.dx[a] = 2.0 * m->lv.back().dx[a];
      size_t ncg = (size_t)c.L->ncg, ns = (size_t)c.L->nside_tot;
      rc |= talloc(&c.C, ncg);
      rc |= talloc(&c.M, ncg);
      rc |= talloc(&c.D, ns);
      rc |= talloc(&c.fc, ns);
      rc |= talloc(&c.sm, ncg);
      rc |= talloc(&c.x, (size_t)ncomp_max * ncg);
      rc |= talloc(&c.b, (size_t)ncomp_max * ncg);
      rc |= talloc(&c.r, checker_ok(*c.L) ? 1 : (size_t)ncomp_max * ncg);
      m->lv.push_back(c);
   }
   if (rc) {
      set_error("mg_create: out of device memory");
      mg_destroy(m);
      return -1;
   }
   *out = m;
   return 0;
}

template <typename T>
void mg_destroy(Mg<T>* m)
{
   if (!m) return;
   for (size_t l = 0; l < m->lv.size(); l++) {
      MgLevel<T>& c = m->lv[l];
      (void)hipFree(c.r);
      if (l == 0) continue;
      (void)hipFree(c.C);
      (void)hipFree(c.M);
      (void)hipFree(c.D);
      (void)hipFree(c.fc);
      (void)hipFree(c.sm);
      (void)hipFree(c.x);
      (void)hipFree(c.b);
      level_destroy(c.L);
   }
   delete m;
}

template <typename T>
int mg_setup_phase(Mg<T>& m, const T* C0, const T* M0, hipStream_t s)
{
   for (int l = 1; l < m.nlev(); l++) {
      const T* f = l == 1 ? C0 : m.lv[l - 1].C;
      if (mg_restrict_cell<T>(*m.lv[l].L, *m.lv[l - 1].L, 1, f, m.lv[l].C, s)) return -1;
      if (M0) {
         const T* fm = l == 1 ? M0 : m.lv[l - 1].M;
         if (mg_restrict_cell<T>(*m.lv[l].L, *m.lv[l - 1].L, 1, fm, m.lv[l].M, s)) return -1;
      }
   }
   return 0;
}

template <typename T>
int mg_setup_conc(Mg<T>& m, const T* D0, hipStream_t s)
{
   for (int l = 1; l < m.nlev(); l++) {
      const T* f = l == 1 ? D0 : m.lv[l - 1].D;
      if (mg_restrict_side<T>(*m.lv[l].L, *m.lv[l - 1].L, f, m.lv[l].D, s)) return -1;
   }
   return 0;
}

template <typename T>
int mg_setup_quat(Mg<T>& m, const T* fc0, const T* sm0, hipStream_t s)
{
   for (int l = 1; l < m.nlev(); l++) {
      const Level& C = *m.lv[l].L;
      const Level& F = *m.lv[l - 1].L;
      const T* ff = l == 1 ? fc0 : m.lv[l - 1].fc;
      const T* fs = l == 1 ? sm0 : m.lv[l - 1].sm;
      if (mg_restrict_side<T>(C, F, ff, m.lv[l].fc, s)) return -1;
      if (mg_restrict_cell<T>(C, F, 1, fs, m.lv[l].sm, s)) return -1;
      if (ghost_fill(C, m.lv[l].sm, 1, s)) return -1;
   }
   return 0;
}

// ------------------------------------------------------------ cycles
// The residual after red-black sweeps ending with the black colour vanishes
// on black cells when every black cell's neighbours are red (checker_ok: a
// zero-slope ghost, at a bounded side or next to cells no patch covers, copies a
// cell's own value into its row).  One, two or four components.
bool red_residual_ok(const Level& L, int ncomp)
{
   return checker_ok(L) && (ncomp == 1 || ncomp == 2 || ncomp == 4);
}

// The set's operators on level l.
template <typename T>
static SweepSet<T> level_set(const Mg<T>& m, const SweepSet<T>& set, int l)
{
   SweepSet<T> r = set;
   if (l == 0) return r;
   const MgLevel<T>& c = m.lv[l];
   for (int i = 0; i < r.n; i++) {
      SweepSlot<T>& o = r.s[i];
      o.b = nullptr;
      if (o.kind == 1) {
         o.D = c.fc;
         o.sm = c.sm;
      } else if (o.D) {
         o.D = c.D;
      } else {
         o.C = c.C;
         if (o.M) o.M = c.M;
      }
   }
   return r;
}

// Red-black sweeps of a set on a level.  zero: x holds nothing yet and stands for
// zero.  On one checkerboard the first two colours then start from what they
// know (SetForm::from) and nothing is cleared; elsewhere a colour may read its
// own colour across the boundary, and x is cleared.  A level that wraps fills
// no ghosts.
template <typename T>
int set_smooth(const Level& L, const SweepSet<T>& set, const double* dx, int ncomp, const T* b,
               T* x, int sweeps, bool zero, bool split, hipStream_t s)
{
   const bool wrap = level_wrap_ok(L), ck = checker_ok(L);
   if (zero && (!ck || sweeps == 0) && fill_zero<T>(x, L.ncg * ncomp, s)) return -1;
   SetForm form;
   form.split = split;
   form.wrap = wrap;
   for (int c = 0; c < 2 * sweeps; c++) {
      form.from = zero && ck && c < 2 ? 1 + c : 0;
      if (!wrap && !(zero && c == 0) && ghost_fill_faces(L, x, ncomp, s, split)) return -1;
      if (launch_set_sweep<T>(L, set, dx, b, x, c & 1, form, s)) return -1;
   }
   return 0;
}
template int set_smooth<float>(const Level&, const SweepSet<float>&, const double*, int,
                               const float*, float*, int, bool, bool, hipStream_t);
template int set_smooth<double>(const Level&, const SweepSet<double>&, const double*, int,
                                const double*, double*, int, bool, bool, hipStream_t);

template <typename T>
int mg_vcycle(Mg<T>& m, const SweepSet<T>& set, const MgCycle& cy, const T* b0, T* x0, bool split,
              hipStream_t s)
{
   int nc = 0;
   for (int i = 0; i < set.n; i++) nc += set.s[i].ncomp;
   if (nc > m.ncomp_max || (split && !m.split)) {
      set_error("mg_vcycle: more components than the hierarchy holds, or no split tables");
      return -1;
   }
   const int nl = m.nlev();
   SetForm form;
   form.split = split;
   for (int l = 0; l < nl; l++) {
      MgLevel<T>& c = m.lv[l];
      const T* b = l == 0 ? b0 : c.b;
      T* x = l == 0 ? x0 : c.x;
      const SweepSet<T> ls = level_set(m, set, l);
      const int nu = l == nl - 1 ? cy.ncoarse : cy.nu1;
      if (set_smooth<T>(*c.L, ls, c.dx, nc, b, x, nu, true, split, s)) return -1;
      if (l == nl - 1) break;
      MgLevel<T>& n = m.lv[l + 1];
      form.wrap = level_wrap_ok(*c.L);
      if (!form.wrap && ghost_fill_faces(*c.L, x, nc, s, split)) return -1;
      if (nu >= 1 && checker_ok(*c.L)) {
         // the sweeps end with the black colour: restrict the red residuals
         if (launch_set_resrestrict<T>(*n.L, *c.L, ls, c.dx, b, x, n.b, form, s)) return -1;
      } else {
         // (a checkerboard level without sweeps: x is zero, the residual is b)
         const T* r = checker_ok(*c.L) ? b : c.r;
         if (r != b && launch_set_residual<T>(*c.L, ls, c.dx, b, x, c.r, split, s)) return -1;
         if (mg_restrict_cell<T>(*n.L, *c.L, nc, r, n.b, s, split)) return -1;
      }
   }
   for (int l = nl - 2; l >= 0; l--) {
      MgLevel<T>& c = m.lv[l];
      MgLevel<T>& n = m.lv[l + 1];
      const T* b = l == 0 ? b0 : c.b;
      T* x = l == 0 ? x0 : c.x;
      // the interpolation reads edge and corner ghosts too
      const bool wrap = level_wrap_ok(*n.L);
      if (!wrap && ghost_fill(*n.L, n.x, nc, s, split)) return -1;
      if (mg_prolong_add<T>(*c.L, *n.L, nc, 1, n.x, x, s, split, wrap)) return -1;
      if (set_smooth<T>(*c.L, level_set(m, set, l), c.dx, nc, b, x, cy.nu2, false, split, s))
         return -1;
   }
   return 0;
}

template <typename T>
int mg_enable_split(Mg<T>& m, hipStream_t s)
{
   for (auto& c : m.lv)
      if (level_split_tables(*c.L, s)) return -1;
   m.split = true;
   return 0;
}

#define AMPE_MG_INST(T)                                                                      \
   template int mg_create<T>(const Level&, const double*, int, int, int, Mg<T>**);          \
   template void mg_destroy<T>(Mg<T>*);                                                      \
   template int mg_setup_phase<T>(Mg<T>&, const T*, const T*, hipStream_t);                  \
   template int mg_setup_conc<T>(Mg<T>&, const T*, hipStream_t);                             \
   template int mg_setup_quat<T>(Mg<T>&, const T*, const T*, hipStream_t);                   \
   template int mg_vcycle<T>(Mg<T>&, const SweepSet<T>&, const MgCycle&, const T*, T*, bool,  \
                             hipStream_t);                                                   \
   template int mg_restrict_cell<T>(const Level&, const Level&, int, const T*, T*,           \
                                    hipStream_t, bool);                                      \
   template int mg_restrict_side<T>(const Level&, const Level&, const T*, T*, hipStream_t);  \
   template int mg_prolong_add<T>(const Level&, const Level&, int, int, const T*, T*,        \
                                  hipStream_t, bool, bool);
AMPE_MG_INST(float)
AMPE_MG_INST(double)
template int mg_enable_split<float>(Mg<float>&, hipStream_t);

}  // namespace ampe
