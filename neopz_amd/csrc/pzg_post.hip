// pzg_post.hip -- post-processing of the device solution.
//
//  * k_post<NS, POINTS>: the error norms of TPZInterpolationSpace::
//    EvaluateError (Mesh/pzinterpolationspace.cpp:1108-1207): per volume
//    element the weighted sum over the error rule's points of the material's
//    Errors values, then its square root.  A group of G lanes (G = the power
//    of two >= the rule's point count, at most 64) takes EB elements: their
//    solution coefficients, table columns and corner coordinates go to LDS
//    (sides without equations are left out), each lane walks the points q =
//    lane, lane + G, ... of tables stored point-fastest (coalesced loads), and
//    the group adds its lanes' sums with cross-lane shuffles.  With POINTS = true the kernel writes the
//    physical coordinates of the points instead (the points at which a
//    caller evaluates its exact-solution function).
//
// Elements of one rule bucket share one table; a launch covers one bucket.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "pzg_internal.h"

namespace pzg {

constexpr int PTPB = 256;
constexpr int MAXERR = 6;

struct PostArgs {
  const double *xyz;
  const int64_t *nodes, *conn, *aidx, *off;
  const int32_t *list, *slot;  // slot: col_off[HP_MAXSH] | side[HP_MAXSH]
  const double *coef, *u, *tab, *uq, *duq;
  const int64_t *dep_ptr, *dep_blk;  // constrained connects (may be null)
  const double *dep_coef;
  double *out, *xq;
  int64_t nlist;
  int nq, ncol, nslot, nsv, nc, dim, bs, G, hp, tet, material, kind, nerr;
  double center[3], cst, E, nu, kconst;
};

// Scalar exact solutions of TLaplaceExample1::uxy (Pre/TPZAnalyticSolution.
// cpp:1254-1310) and their gradients (graduxy, :1927-1943, by automatic
// differentiation there, in closed form here).
__device__ inline void exact_dev(const PostArgs &a, const double x[3], double &ue, double ge[3]) {
  const double PI = 3.14159265358979323846;
  const double xl[3] = {x[0] - a.center[0], x[1] - a.center[1], x[2] - a.center[2]};
  ge[0] = ge[1] = ge[2] = 0.;
  ue = 0.;
  if (a.kind == PZG_EXACT_CONST) {
    ue = a.cst;
  } else if (a.kind == PZG_EXACT_X) {
    ue = xl[0];
    ge[0] = 1.;
  } else {
    const bool sn = a.kind == PZG_EXACT_SINSIN;
    double f[3], df[3];
    for (int i = 0; i < a.dim; i++) {
      double s, c;
      if (sn) {
        sincos(PI * xl[i], &s, &c);
        f[i] = s;
        df[i] = PI * c;
      } else {
        sincos(PI * xl[i] / 2, &s, &c);
        f[i] = c;
        df[i] = -(PI / 2) * s;
      }
    }
    ue = 1.;
    for (int i = 0; i < a.dim; i++) ue *= f[i];
    for (int j = 0; j < a.dim; j++) {
      double g = df[j];
      for (int i = 0; i < a.dim; i++)
        if (i != j) g *= f[i];
      ge[j] = g;
    }
  }
}

// The materials' Errors at one point; u/g: discrete value and gradient
// (g[i][k] = d u_k / d x_i), ue/ge the exact ones.
//   TPZMatPoisson::Errors (Material/Poisson/TPZMatPoisson.cpp:173-218)
//   TPZDarcyFlow::Errors (Material/DarcyFlow/TPZDarcyFlow.cpp:268-326): the
//     semi-norm term is (sum_i K |g_i - ge_i|)^2 and the flux terms compare
//     the exact derivative with -K g, as written there
//   TPZElasticity3D::Errors (Material/Elasticity/TPZElasticity3D.cpp:
//     1081-1133) with ComputeStressVector (:1178-1192), no prestress
template <int NS>
__device__ inline void err_values(const PostArgs &a, double coef, const double (&u)[NS],
                                  const double (&g)[3][NS], const double (&ue)[NS],
                                  const double (&ge)[3][NS], double (&v)[MAXERR]) {
  for (int m = 0; m < MAXERR; m++) v[m] = 0.;
  if constexpr (NS == 1) {
    if (a.material == PZG_MAT_POISSON) {
      const double d = u[0] - ue[0];
      v[1] = d * d;
      for (int i = 0; i < a.dim; i++) {
        const double t = g[i][0] - ge[i][0];
        v[2] += t * t;
      }
      v[0] = v[1] + v[2];
    } else {
      const double d = fabs(u[0] - ue[0]);
      v[1] = d * d;
      double s = 0.;
      for (int i = 0; i < a.dim; i++) s += coef * fabs(g[i][0] - ge[i][0]);
      v[2] = fabs(s * s);
      v[0] = v[1] + v[2];
      for (int i = 0; i < a.dim; i++) {
        const double t = fabs(ge[i][0] - (-coef * g[i][0]));
        v[3 + i] = t * t;
      }
    }
  } else {
    double l2 = 0., semi = 0., D[3][3];
    for (int k = 0; k < 3; k++) l2 += (u[k] - ue[k]) * (u[k] - ue[k]);
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) {
        D[i][j] = g[i][j] - ge[i][j];
        semi += D[i][j] * D[i][j];
      }
    const double E = coef, ni = a.nu;
    const double c1 = -1. + ni, c2 = -1. + ni + 2. * ni * ni, c3 = 2. * (1. + ni);
    const double s0 = E * (D[0][0] * c1 - (D[1][1] + D[2][2]) * ni) / c2;
    const double s1 = E * (D[1][1] * c1 - (D[0][0] + D[2][2]) * ni) / c2;
    const double s2 = E * (D[2][2] * c1 - (D[0][0] + D[1][1]) * ni) / c2;
    const double s3 = E * (D[1][0] + D[0][1]) / c3;
    const double s4 = E * (D[2][0] + D[0][2]) / c3;
    const double s5 = E * (D[2][1] + D[1][2]) / c3;
    const double S[3][3] = {{s0, s3, s4}, {s3, s1, s5}, {s4, s5, s2}};
    double en = 0.;
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) en += D[i][j] * S[i][j];
    v[0] = en;
    v[1] = l2;
    v[2] = semi;
  }
}

// g = (gradient in x, y, z) of the reference gradient gr, and |det J| (the element's
// volume / area / length measure) (Axes2XYZ of the axes gradient); dim 3: ji[d][i]
// = d xi_d / d x_i
__device__ inline double jac_inverse(const double (&J)[3][3], double (&ji)[3][3]) {
  const double det = -J[0][2] * J[1][1] * J[2][0] + J[0][1] * J[1][2] * J[2][0] + J[0][2] * J[1][0] * J[2][1] -
                     J[0][0] * J[1][2] * J[2][1] - J[0][1] * J[1][0] * J[2][2] + J[0][0] * J[1][1] * J[2][2];
  ji[0][0] = (-J[1][2] * J[2][1] + J[1][1] * J[2][2]) / det;
  ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) / det;
  ji[0][2] = (-J[0][2] * J[1][1] + J[0][1] * J[1][2]) / det;
  ji[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) / det;
  ji[1][1] = (-J[0][2] * J[2][0] + J[0][0] * J[2][2]) / det;
  ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) / det;
  ji[2][0] = (-J[1][1] * J[2][0] + J[1][0] * J[2][1]) / det;
  ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) / det;
  ji[2][2] = (-J[0][1] * J[1][0] + J[0][0] * J[1][1]) / det;
  return det;
}

// EB elements per group of lanes share every table value it loads; AFF:
// tetrahedra, whose Jacobian is the same at every point (the corner derivatives
// are -1, 0, 1) and is inverted once per element.
//
// One element per group was bound by the L1: four table values for four
// multiply-adds, over all 56 sides of an order-5 element whatever its order.
// 82,944 tetrahedra of orders 1 to 5, 512 points each: 8.57 ms of kernels then,
// 2.3 now with EB = 4 (247 registers, two wavefronts per SIMD); with EB = 2 the
// call takes 0.08 ms more.  What is left is arithmetic: the exact solution's
// sines and the multiply-adds.
template <int NS, bool POINTS, int EB, bool AFF>
__global__ __launch_bounds__(PTPB) void k_post(const PostArgs a) {
  extern __shared__ double s_mem[];
  const int G = a.G, ngrp = PTPB / G;
  const int gl = threadIdx.x / G, lq = threadIdx.x - gl * G;
  const int64_t g0 = ((int64_t)blockIdx.x * ngrp + gl) * EB;
  const bool live = g0 < a.nlist;
  int64_t e[EB];
#pragma unroll
  for (int j = 0; j < EB; j++) e[j] = live ? a.list[g0 + j < a.nlist ? g0 + j : a.nlist - 1] : 0;
  const int gsz = a.nslot * NS * EB + (24 + (AFF ? 10 : 0)) * EB;
  double *s_u = s_mem + (size_t)gl * gsz;  // [slot][state][element]
  double *s_x = s_u + a.nslot * NS * EB;   // corners, then det and ji
  double *s_j = s_x + 24 * EB;
  int *s_col = reinterpret_cast<int *>(s_mem + (size_t)ngrp * gsz) + gl * a.nslot * EB;
  const int nc = a.nc, dim = a.dim, nq = a.nq, ncol = a.ncol;
  const double *W = a.tab, *PH = W + nq, *DPH = PH + (size_t)ncol * nq;
  const double *CP = DPH + (size_t)dim * ncol * nq, *CD = CP + (size_t)nc * nq;
  int nact = 0;  // slots with a value in one of the elements
  if (live) {
    const int sh = threadIdx.x & 63 & ~(G - 1);
    const uint64_t below = (1ull << lq) - 1, mine = G < 64 ? (1ull << G) - 1 : ~0ull;
    if (!POINTS)
      for (int i0 = 0; i0 < a.nslot; i0 += G) {
        const int i = i0 + lq;
        double v[EB][NS];
        int col[EB], c0 = 0;
        bool any = false, differ = false;
#pragma unroll
        for (int j = 0; j < EB; j++) {
          col[j] = 0;
#pragma unroll
          for (int k = 0; k < NS; k++) v[j][k] = 0.;
          if (i >= a.nslot) continue;
          // a constrained connect's value follows from the connects it depends
          // on (TPZCompMesh::LoadSolution expands the solution)
          const int64_t cc = a.conn[e[j] * a.nsv + i], b = a.aidx[cc];
          const bool has = b >= 0 || a.dep_ptr;
          if (!has) continue;  // no equations: no term
          for (int k = 0; k < NS; k++) {
            if (b >= 0) v[j][k] = a.u[b * a.bs + k];
            else
              for (int64_t d = a.dep_ptr[cc]; d < a.dep_ptr[cc + 1]; d++)
                if (a.dep_blk[d] >= 0) v[j][k] += a.dep_coef[d] * a.u[a.dep_blk[d] * a.bs + k];
          }
          col[j] = i;
          if (a.hp) {
            int64_t id[4] = {0, 0, 0, 0};
            for (int k = 0; k < nc; k++) id[k] = a.nodes[e[j] * nc + k];
            col[j] = a.slot[i] + hp_variant(a.tet, a.slot[HP_MAXSH + i], id);
          }
          if (!any) c0 = col[j];
          else differ |= col[j] != c0;
          any = true;
        }
        const uint64_t m = (__ballot(any) >> sh) & mine;
        if (any) {
          const int at = nact + __popcll(m & below);
#pragma unroll
          for (int j = 0; j < EB; j++) {
#pragma unroll
            for (int k = 0; k < NS; k++) s_u[(at * NS + k) * EB + j] = v[j][k];
            // negative: the elements' columns differ
            if (j > 0 || !differ) s_col[at * EB + j] = differ ? col[j] : c0;
          }
          if (differ) s_col[at * EB] = -1 - col[0];
        }
        nact += __popcll(m);
      }
#pragma unroll
    for (int j = 0; j < EB; j++)
      for (int k = lq; k < nc * 3; k += G) s_x[j * 24 + k] = a.xyz[3 * a.nodes[e[j] * nc + k / 3] + k % 3];
  }
  __syncthreads();
  if (AFF) {
    for (int j = lq; live && j < EB; j += G) {
      double J[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}}, ji[3][3];
      for (int n = 0; n < nc; n++)
        for (int d = 0; d < 3; d++) {
          const double cd = CD[((size_t)d * nc + n) * nq];
          for (int i = 0; i < 3; i++) J[i][d] += cd * s_x[j * 24 + 3 * n + i];
        }
      s_j[j * 10] = jac_inverse(J, ji);
      for (int d = 0; d < 3; d++)
        for (int i = 0; i < 3; i++) s_j[j * 10 + 1 + 3 * d + i] = ji[d][i];
    }
    __syncthreads();
  }
  if (!live) return;

  double acc[EB][MAXERR];
#pragma unroll
  for (int j = 0; j < EB; j++)
#pragma unroll
    for (int m = 0; m < MAXERR; m++) acc[j][m] = 0.;
  for (int q = lq; q < nq; q += G) {
    // discrete value and reference gradient (TPZInterpolationSpace::
    // ComputeSolution)
    double u[EB][NS], gr[EB][3][NS];
#pragma unroll
    for (int j = 0; j < EB; j++)
#pragma unroll
      for (int k = 0; k < NS; k++) {
        u[j][k] = 0.;
        for (int d = 0; d < 3; d++) gr[j][d][k] = 0.;
      }
    for (int i = 0; i < nact; i++) {
      const int col = s_col[i * EB];
      if (EB == 1 || col >= 0) {
        const double ph = PH[(size_t)col * nq + q];
        double dp[3] = {0., 0., 0.};
#pragma unroll
        for (int d = 0; d < 3; d++)
          if (d < dim) dp[d] = DPH[((size_t)d * ncol + col) * nq + q];
#pragma unroll
        for (int k = 0; k < NS; k++)
#pragma unroll
          for (int j = 0; j < EB; j++) {
            const double cf = s_u[(i * NS + k) * EB + j];
            u[j][k] += ph * cf;
#pragma unroll
            for (int d = 0; d < 3; d++) gr[j][d][k] += dp[d] * cf;
          }
      } else {
#pragma unroll
        for (int j = 0; j < EB; j++) {
          const int cj = j == 0 ? -1 - col : s_col[i * EB + j];
          const double ph = PH[(size_t)cj * nq + q];
          double dp[3] = {0., 0., 0.};
#pragma unroll
          for (int d = 0; d < 3; d++)
            if (d < dim) dp[d] = DPH[((size_t)d * ncol + cj) * nq + q];
#pragma unroll
          for (int k = 0; k < NS; k++) {
            const double cf = s_u[(i * NS + k) * EB + j];
            u[j][k] += ph * cf;
#pragma unroll
            for (int d = 0; d < 3; d++) gr[j][d][k] += dp[d] * cf;
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < EB; j++) {
      // geometric map: x and J[i][d] = d x_i / d xi_d (TPZGeoEl::X / GradX)
      double x[3] = {0., 0., 0.}, J[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}};
      for (int n = 0; n < nc; n++) {
        const double cp = CP[(size_t)n * nq + q];
#pragma unroll
        for (int i = 0; i < 3; i++) x[i] += cp * s_x[j * 24 + 3 * n + i];
        if (!AFF)
#pragma unroll
          for (int d = 0; d < 3; d++)
            if (d < dim) {
              const double cd = CD[((size_t)d * nc + n) * nq + q];
#pragma unroll
              for (int i = 0; i < 3; i++) J[i][d] += cd * s_x[j * 24 + 3 * n + i];
            }
      }
      if constexpr (POINTS) {
        const int64_t p = a.off[e[j]] + q;
        for (int i = 0; i < 3; i++) a.xq[p * 3 + i] = x[i];
        continue;
      }
      double g[3][NS], det;
      if (AFF || dim == 3) {
        double ji[3][3];
        if (AFF) {
          det = s_j[j * 10];
#pragma unroll
          for (int d = 0; d < 9; d++) ji[d / 3][d % 3] = s_j[j * 10 + 1 + d];
        } else {
          det = jac_inverse(J, ji);
        }
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
          for (int k = 0; k < NS; k++)
            g[i][k] = ji[0][i] * gr[j][0][k] + ji[1][i] * gr[j][1][k] + ji[2][i] * gr[j][2][k];
      } else if (dim == 2) {
        // surface element: g = J (J^T J)^-1 grad_xi, det = sqrt(det J^T J)
        const double g11 = J[0][0] * J[0][0] + J[1][0] * J[1][0] + J[2][0] * J[2][0];
        const double g12 = J[0][0] * J[0][1] + J[1][0] * J[1][1] + J[2][0] * J[2][1];
        const double g22 = J[0][1] * J[0][1] + J[1][1] * J[1][1] + J[2][1] * J[2][1];
        const double dg = g11 * g22 - g12 * g12;
        det = sqrt(dg);
        for (int k = 0; k < NS; k++) {
          const double h0 = (g22 * gr[j][0][k] - g12 * gr[j][1][k]) / dg;
          const double h1 = (-g12 * gr[j][0][k] + g11 * gr[j][1][k]) / dg;
          for (int i = 0; i < 3; i++) g[i][k] = J[i][0] * h0 + J[i][1] * h1;
        }
      } else {
        const double l2 = J[0][0] * J[0][0] + J[1][0] * J[1][0] + J[2][0] * J[2][0];
        det = sqrt(l2);
        for (int k = 0; k < NS; k++)
          for (int i = 0; i < 3; i++) g[i][k] = J[i][0] * gr[j][0][k] / l2;
      }
      // exact solution at x
      double ue[NS], ge[3][NS];
      if (a.kind == PZG_EXACT_POINTS) {
        const int64_t p = a.off[e[j]] + q;
        for (int k = 0; k < NS; k++) {
          ue[k] = a.uq[p * NS + k];
          for (int d = 0; d < 3; d++) ge[d][k] = d < dim ? a.duq[(p * dim + d) * NS + k] : 0.;
        }
      } else {
        double g1[3], u1;
        exact_dev(a, x, u1, g1);
        for (int k = 0; k < NS; k++) {
          ue[k] = u1;
          for (int d = 0; d < 3; d++) ge[d][k] = g1[d];
        }
      }
      const double coef = a.coef ? a.coef[e[j]] : (a.material == PZG_MAT_ELAST3D ? a.E : a.kconst);
      double v[MAXERR];
      err_values<NS>(a, coef, u[j], g, ue, ge, v);
      const double wdet = W[q] * fabs(det);
#pragma unroll
      for (int m = 0; m < MAXERR; m++) acc[j][m] += wdet * v[m];
      __builtin_amdgcn_sched_barrier(0);  // one element at a time (else 256 registers for four)
    }
  }
  if constexpr (POINTS) return;
#pragma unroll
  for (int j = 0; j < EB; j++) {
    for (int o = G >> 1; o > 0; o >>= 1)
#pragma unroll
      for (int m = 0; m < MAXERR; m++) acc[j][m] += __shfl_xor(acc[j][m], o, 64);
    if (lq == 0 && g0 + j < a.nlist)
#pragma unroll
      for (int m = 0; m < MAXERR; m++)
        if (m < a.nerr) a.out[e[j] * a.nerr + m] = sqrt(acc[j][m]);
  }
}

// ---------------------------------------------------------------------------
// Error-rule tables of every rule bucket for an exact solution of order
// porder, the element lists of the buckets and the point offsets.
static int post_prepare(Ctx &c, int porder) {
  if (!c.has_mesh) {
    set_error("post-processing: no mesh");
    return PZG_ESTATE;
  }
  if (porder < 0 || porder > 1000) {
    set_error("post-processing: exact-solution order out of range");
    return PZG_EINVAL;
  }
  if (c.post_porder == porder) return PZG_OK;
  const int nbk = (int)c.vol_rules.size();
  const bool hp = c.hp_simplex;
  c.post_tab.assign(nbk, PostTables());
  std::vector<int32_t> slot((size_t)nbk * 2 * HP_MAXSH, 0);
  c.post_tab_off.assign(nbk + 1, 0);
  for (int b = 0; b < nbk; b++) {
    const int order = post_rule_order(c.vol_etype, c.vol_rules[b], porder);
    PostTables &t = c.post_tab[b];
    PZG_TRY(build_post_tables(c.vol_etype, hp ? c.hp_order : c.porder, hp, order, t));
    if (hp && t.nsh != c.vol_nsides) {
      set_error("post-processing: virtual sides do not match the shape list");
      return PZG_EINVAL;
    }
    for (int i = 0; i < t.nsh; i++) {
      slot[(size_t)b * 2 * HP_MAXSH + i] = t.col_off[i];
      slot[(size_t)b * 2 * HP_MAXSH + HP_MAXSH + i] = t.shape_side[i];
    }
    c.post_tab_off[b + 1] = c.post_tab_off[b] + (int64_t)t.d.size();
  }
  std::vector<double> tab(c.post_tab_off[nbk]);
  for (int b = 0; b < nbk; b++)
    std::memcpy(tab.data() + c.post_tab_off[b], c.post_tab[b].d.data(),
                c.post_tab[b].d.size() * sizeof(double));
  std::vector<int64_t> off(c.nvol + 1, 0);
  c.post_lptr.assign(nbk + 1, 0);
  for (int64_t e = 0; e < c.nvol; e++) {
    off[e + 1] = off[e] + c.post_tab[c.vol_bucket[e]].nq;
    c.post_lptr[c.vol_bucket[e] + 1]++;
  }
  for (int b = 0; b < nbk; b++) c.post_lptr[b + 1] += c.post_lptr[b];
  std::vector<int32_t> list(c.nvol);
  {
    std::vector<int64_t> fill(c.post_lptr.begin(), c.post_lptr.end() - 1);
    if (hp) {
      // elements whose vertex ids are in the same order have the same table
      // columns and come next to each other
      std::vector<uint8_t> key(c.nvol);
      int64_t cnt[257] = {0};
      for (int64_t e = 0; e < c.nvol; e++) {
        const int64_t *id = &c.vol_nodes[e * c.vol_ncorner];
        int k = 0;
        for (int i = 0; i < c.vol_ncorner; i++)
          for (int j = 0; j < i; j++) k = 2 * k + (id[j] < id[i] ? 1 : 0);
        key[e] = (uint8_t)k;  // at most 6 comparisons
        cnt[k + 1]++;
      }
      for (int k = 0; k < 256; k++) cnt[k + 1] += cnt[k];
      std::vector<int32_t> byk(c.nvol);
      for (int64_t e = 0; e < c.nvol; e++) byk[cnt[key[e]]++] = (int32_t)e;
      for (int64_t k = 0; k < c.nvol; k++) list[fill[c.vol_bucket[byk[k]]]++] = byk[k];
    } else {
      for (int64_t e = 0; e < c.nvol; e++) list[fill[c.vol_bucket[e]]++] = (int32_t)e;
    }
  }
  hipStream_t s = c.stream;
  PZG_TRY(dev_upload(c.d_post_tab, tab.data(), tab.size(), s));
  PZG_TRY(dev_upload(c.d_post_list, list.data(), list.size(), s));
  PZG_TRY(dev_upload(c.d_post_off, off.data(), off.size(), s));
  PZG_TRY(dev_upload(c.d_post_slot, slot.data(), slot.size(), s));
  PZG_HIP(hipStreamSynchronize(s));
  c.post_npts = off[c.nvol];
  c.post_porder = porder;
  return PZG_OK;
}

// One launch per rule bucket.
template <bool POINTS>
static int post_launch(Ctx &c, PostArgs a) {
  const bool hp = c.hp_simplex;
  for (size_t b = 0; b + 1 < c.post_lptr.size(); b++) {
    const PostTables &t = c.post_tab[b];
    a.nlist = c.post_lptr[b + 1] - c.post_lptr[b];
    if (a.nlist == 0) continue;
    a.list = c.d_post_list.as<int32_t>() + c.post_lptr[b];
    a.tab = c.d_post_tab.as<double>() + c.post_tab_off[b];
    a.slot = c.d_post_slot.as<int32_t>() + b * 2 * HP_MAXSH;
    a.nq = t.nq;
    a.ncol = t.ncol;
    a.nslot = hp ? t.nsh : (t.ncol < c.vol_nsides ? t.ncol : c.vol_nsides);
    // G lanes per element (a power of two up to a wavefront), enough for the
    // element's points, and enough for the workgroup's elements to fit in LDS
    const bool aff = c.vol_etype == PZG_TET;
    auto lds_of = [&](int g, int eb) {
      return (size_t)(PTPB / g) * eb * ((size_t)a.nslot * (POINTS ? 1 : c.nstate) * 8 + (24 + 10) * 8 + a.nslot * 4);
    };
    auto group = [&](int eb) {
      int G = 1;
      while (G < 64 && (G < t.nq || lds_of(G, eb) > 65536)) G <<= 1;
      return G;
    };
    // elements per group: as many as registers hold, when that still leaves two
    // workgroups per CU (below it, fewer elements per group fill the chip better)
    int eb = POINTS ? 1 : c.nstate == 1 && aff ? 4 : 2;
    if (eb > 1 && (a.nlist < (int64_t)512 * eb * (PTPB / group(eb)) || lds_of(group(eb), eb) > 65536)) eb = 1;
    const int G = group(eb);
    a.G = G;
    const size_t lds = lds_of(G, eb);
    if (lds > 65536) {
      set_error("post-processing: element too large for the error kernel");
      return PZG_EUNSUP;
    }
    const int64_t per = (int64_t)(PTPB / G) * eb;
    const dim3 grid((unsigned)((a.nlist + per - 1) / per));
    if (POINTS) hipLaunchKernelGGL((k_post<1, true, 1, false>), grid, dim3(PTPB), lds, c.stream, a);
    else if (c.nstate == 1 && eb == 4) hipLaunchKernelGGL((k_post<1, false, 4, true>), grid, dim3(PTPB), lds, c.stream, a);
    else if (c.nstate == 1 && eb == 2) hipLaunchKernelGGL((k_post<1, false, 2, false>), grid, dim3(PTPB), lds, c.stream, a);
    else if (c.nstate == 1) hipLaunchKernelGGL((k_post<1, false, 1, false>), grid, dim3(PTPB), lds, c.stream, a);
    else if (eb == 2) hipLaunchKernelGGL((k_post<3, false, 2, false>), grid, dim3(PTPB), lds, c.stream, a);
    else hipLaunchKernelGGL((k_post<3, false, 1, false>), grid, dim3(PTPB), lds, c.stream, a);
    PZG_HIP(hipGetLastError());
  }
  return PZG_OK;
}

static PostArgs post_args(const Ctx &c) {
  PostArgs a;
  std::memset(&a, 0, sizeof(a));
  a.xyz = c.d_xyz.as<double>();
  a.nodes = c.d_vnodes.as<int64_t>();
  a.conn = c.d_vconn.as<int64_t>();
  a.aidx = c.d_aidx.as<int64_t>();
  a.off = c.d_post_off.as<int64_t>();
  a.coef = c.vol_coef.empty() ? nullptr : c.d_vcoef.as<double>();
  a.nsv = c.vol_nsides;
  a.nc = c.vol_ncorner;
  a.dim = c.dim;
  a.bs = c.bs;
  a.hp = c.hp_simplex ? 1 : 0;
  a.tet = c.vol_etype == PZG_TET ? 1 : 0;
  a.material = c.material;
  a.E = c.E;
  a.nu = c.nu;
  a.kconst = c.scale;
  if (c.has_dep) {
    a.dep_ptr = c.d_dep_ptr.as<int64_t>();
    a.dep_blk = c.d_dep_blk.as<int64_t>();
    a.dep_coef = c.d_dep_coef.as<double>();
  }
  return a;
}

int post_points(Ctx &c, int porder, int64_t *npts, double *xq) {
  PZG_TRY(post_prepare(c, porder));
  if (npts) *npts = c.post_npts;
  if (!xq) return PZG_OK;
  PZG_TRY(dev_alloc(c.d_post_xq, (size_t)c.post_npts * 3 * sizeof(double)));
  PostArgs a = post_args(c);
  a.xq = c.d_post_xq.as<double>();
  PZG_TRY(post_launch<true>(c, a));
  PZG_HIP(hipMemcpyAsync(xq, c.d_post_xq.p, (size_t)c.post_npts * 3 * sizeof(double),
                         hipMemcpyDeviceToHost, c.stream));
  PZG_HIP(hipStreamSynchronize(c.stream));
  return PZG_OK;
}

int post_errors(Ctx &c, const pzg_exact &ex, double *el_errors, double *errors, int *nerr_out) {
  if (!c.has_mesh) {
    set_error("pzg_evaluate_error: no mesh");
    return PZG_ESTATE;
  }
  if (!c.has_solution) {
    set_error("pzg_evaluate_error: no solution loaded (pzg_solve or pzg_load_solution)");
    return PZG_ESTATE;
  }
  const int nerr = c.material == PZG_MAT_DARCY ? 6 : 3;
  if (ex.kind < PZG_EXACT_POINTS || ex.kind > PZG_EXACT_COSCOS) {
    set_error("pzg_evaluate_error: unknown exact-solution kind");
    return PZG_EINVAL;
  }
  if (ex.kind != PZG_EXACT_POINTS && c.nstate != 1) {
    set_error("pzg_evaluate_error: the device exact solutions are scalar; use PZG_EXACT_POINTS");
    return PZG_EINVAL;
  }
  PZG_TRY(post_prepare(c, ex.porder));
  PostArgs a = post_args(c);
  a.kind = ex.kind;
  a.nerr = nerr;
  for (int d = 0; d < 3; d++) a.center[d] = ex.center[d];
  a.cst = ex.constant;
  hipStream_t s = c.stream;
  if (ex.kind == PZG_EXACT_POINTS) {
    if (ex.npts != c.post_npts || !ex.u || !ex.du) {
      set_error("pzg_evaluate_error: exact values must cover the " + std::to_string(c.post_npts) +
                " points of pzg_error_points for this order");
      return PZG_EINVAL;
    }
    const size_t nu = (size_t)c.post_npts * c.nstate, ndu = nu * c.dim;
    PZG_TRY(dev_upload(c.d_post_uq, ex.u, nu, s));
    PZG_TRY(dev_upload(c.d_post_duq, ex.du, ndu, s));
    a.uq = c.d_post_uq.as<double>();
    a.duq = c.d_post_duq.as<double>();
  }
  a.u = c.d_u.as<double>();
  PZG_TRY(dev_alloc(c.d_post_out, (size_t)c.nvol * nerr * sizeof(double)));
  a.out = c.d_post_out.as<double>();
  PZG_TRY(post_launch<false>(c, a));
  std::vector<double> el((size_t)c.nvol * nerr);
  PZG_HIP(hipMemcpyAsync(el.data(), c.d_post_out.p, el.size() * sizeof(double), hipMemcpyDeviceToHost,
                         s));
  PZG_HIP(hipStreamSynchronize(s));
  // TPZCompMesh::EvaluateError: sum of the squared element norms in element
  // order, then the square root (Mesh/pzcmesh.cpp:1497-1552)
  if (errors) {
    double tot[MAXERR] = {0., 0., 0., 0., 0., 0.};
    for (int64_t e = 0; e < c.nvol; e++)
      for (int m = 0; m < nerr; m++) tot[m] += el[e * nerr + m] * el[e * nerr + m];
    for (int m = 0; m < nerr; m++) errors[m] = std::sqrt(tot[m]);
  }
  if (el_errors) std::memcpy(el_errors, el.data(), el.size() * sizeof(double));
  if (nerr_out) *nerr_out = nerr;
  return PZG_OK;
}

}  // namespace pzg
