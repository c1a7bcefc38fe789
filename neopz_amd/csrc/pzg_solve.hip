// pzg_solve.hip -- gfx950 kernels and drivers of the solve phase.
//
//  PCG64 (plain path, reference semantics).  CG<> of
//  Solvers/LinearSolvers/cg.h:29-132 with the EJacobi TPZStepSolver
//  (z = r / diag, Matrix/pzmatrix.cpp:642-667), x0 = 0, stop on the recursive
//  ||r||/||b|| <= tol.  The reference's Jacobi step also runs a residual SpMV
//  whose result it discards; it has no effect on the iterates and is not run.
//  Matrix: full (both triangles) block CSR of nstate x nstate blocks, FP64
//  values, int32 block columns, expanded once per assembly from the
//  reference upper CSR.
//
//  MIXED.  FP32 flexible CG (Notay's FCG(1)) on S = D^-1/2 K D^-1/2 stored as
//  FP32 block CSR, preconditioned by the inverse diagonal blocks, with FP64
//  reliable updates: whenever the FP32 recursive residual has dropped by a
//  factor delta, the FP32 correction is folded into the FP64 solution
//  (u += D^-1/2 x), the true residual f - K u is recomputed in FP64 and
//  replaces the recursive one, and the iteration continues along the same
//  search direction.  This is iterative refinement (the shape of IR<>,
//  Solvers/LinearSolvers/ir.h:23-66) without restarting the Krylov
//  iteration; the stop test is the true FP64 residual.
//
//  All scalars live on the device; reductions are two-level and
//  deterministic (per-block partials, a one-block kernel sums them in a fixed
//  order), so iterations need no host round trip.  The host only polls the
//  'done' flag once per batch of iterations; a batch can be captured once in
//  a hipGraph and replayed.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>

#include "pzg_device.h"
#include "pzg_internal.h"

namespace pzg {

constexpr int TPB = RED_TPB;

static int grid_for(int64_t n, int per_block) {
  int64_t g = (n + per_block - 1) / per_block;
  if (g > MAXBLK) g = MAXBLK;
  if (g < 1) g = 1;
  return (int)g;
}

// ----------------------------------------------------------------------------
// Block CSR SpMV, shared by the FP64 path (unscaled K) and the FP32 path
// (scaled S).  Every block row is handled by BSR_L lanes; each lane takes
// BSR_U blocks per pass and issues all their loads before the products, so a
// wavefront keeps 64/BSR_L rows x BSR_U blocks of loads in flight.  Values at
// bsr_pos: lane l of a row reads block l of each chunk of BSR_L blocks, the
// chunk component-major, so every value load of the row's lanes is one
// contiguous segment.
#ifndef PZG_BSR_L
#define PZG_BSR_L 16
#endif
#ifndef PZG_BSR_U
#define PZG_BSR_U 4
#endif
constexpr int BSR_L = PZG_BSR_L;
constexpr int BSR_U = PZG_BSR_U;
static_assert(BSR_L == BSR_CHUNK && BSR_L == 16, "a block row is a row of 16 lanes, as the value chunks are");

// xf(i): entry i of the vector.
template <class T, int BS, class X>
__device__ inline void bsr_row_f(int64_t A, const int64_t *__restrict__ bia,
                                 const int32_t *__restrict__ bja, const T *__restrict__ v,
                                 X xf, int sub, T (&out)[BS]) {
  constexpr int BB = BS * BS;
  T acc[BS];
  for (int k = 0; k < BS; k++) acc[k] = T(0);
  const int64_t b0 = bia[A], n = bia[A + 1] - b0;
  for (int64_t base = sub; base < n; base += BSR_L * BSR_U) {
    T m[BSR_U][BB];
    int64_t col[BSR_U];
#pragma unroll
    for (int u = 0; u < BSR_U; u++) {
      const int64_t i = base + BSR_L * u;  // block of the row; i % BSR_L == sub
      if (i < n) {
        col[u] = bja[b0 + i];
        const int64_t j = i - sub, mc = n - j < BSR_L ? n - j : BSR_L;
        const T *vp = v + (b0 + j) * BB + sub;
#pragma unroll
        for (int c = 0; c < BB; c++) m[u][c] = vp[c * mc];
      } else {
        col[u] = 0;
#pragma unroll
        for (int c = 0; c < BB; c++) m[u][c] = T(0);
      }
    }
    T xv[BSR_U][BS];
#pragma unroll
    for (int u = 0; u < BSR_U; u++)
#pragma unroll
      for (int l = 0; l < BS; l++) xv[u][l] = xf(col[u] * BS + l);
#pragma unroll
    for (int u = 0; u < BSR_U; u++)
#pragma unroll
      for (int k = 0; k < BS; k++)
#pragma unroll
        for (int l = 0; l < BS; l++) acc[k] += m[u][k * BS + l] * xv[u][l];
  }
#pragma unroll
  for (int k = 0; k < BS; k++) {
    out[k] = row16_sum(acc[k]);
  }
}

template <class T, int BS>
__device__ inline void bsr_row(int64_t A, const int64_t *__restrict__ bia,
                               const int32_t *__restrict__ bja, const T *__restrict__ v,
                               const T *__restrict__ x, int sub, T (&out)[BS]) {
  bsr_row_f<T, BS>(A, bia, bja, v, [x](int64_t i) { return x[i]; }, sub, out);
}

// lane 'sub' (< BS) of a row group picks component sub of out
template <class T, int BS>
__device__ inline T pick(const T (&out)[BS], int sub) {
  T o = out[0];
#pragma unroll
  for (int k = 1; k < BS; k++)
    if (sub == k) o = out[k];
  return o;
}

// y = A x over block rows; the rows of a workgroup are a contiguous slice
// (xcd_block_range) so that gathers of x stay in one XCD's L2.
template <class T, int BS>
__global__ __launch_bounds__(TPB) void k_spmv_bsr(int64_t nb, const int64_t *__restrict__ bia,
                                                  const int32_t *__restrict__ bja,
                                                  const T *__restrict__ v,
                                                  const T *__restrict__ x, T *__restrict__ y) {
  const int sub = threadIdx.x % BSR_L;
  int64_t lo, hi;
  int xi, xg;
  constexpr int RPB = TPB / BSR_L;  // rows per workgroup tile
#if PZG_XCD_INTERLEAVE
  xcd_slab(nb, lo, hi, xi, xg);
  const int64_t first = lo + (int64_t)xi * RPB, step = (int64_t)xg * RPB;
#else
  xcd_block_range(nb, lo, hi);
  xi = xg = 0;
  const int64_t first = lo, step = RPB;
#endif
  for (int64_t A = first + threadIdx.x / BSR_L; A < hi; A += step) {
    T out[BS];
    bsr_row<T, BS>(A, bia, bja, v, x, sub, out);
    if (sub < BS) y[A * BS + sub] = pick<T, BS>(out, sub);
  }
}

// Sums of NV partial slots, the same bits in every workgroup and thread: each
// workgroup of a step forms the scalars it needs itself, which replaces the
// one-block kernel between two steps (3 to 5 us each on the device, as much as
// a step of a small system).  The step kernels run at most CG_MAXBLK
// workgroups, so the slots stay short.
constexpr int CG_MAXBLK = 512;
template <int NV>
__device__ inline void sum_slots(const double *partials, const int (&slot)[NV], const int (&cnt)[NV],
                                 double (&tot)[NV]) {
  __shared__ double sm[NV][16];
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    double s = 0.;
    for (int b = threadIdx.x; b < cnt[k]; b += blockDim.x) s += partials[slot[k] * MAXBLK + b];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) sm[k][w] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) {
    tot[k] = 0.;
    for (int j = 0; j < nw; j++) tot[k] += sm[k][j];
  }
}

// this workgroup's sums of v into slots 0 .. NV-1 (any workgroup size up to
// 1024)
template <int NV>
__device__ inline void store_slots(const double (&v)[NV], double *partials) {
  __shared__ double sm[NV][16];
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const double s = wave_sum(v[k]);
    if ((threadIdx.x & 63) == 0) sm[k][w] = s;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double s = 0.;
    for (int j = 0; j < nw; j++) s += sm[threadIdx.x][j];
    partials[threadIdx.x * MAXBLK + blockIdx.x] = s;
  }
}

// Workgroup size and grid of the step kernels over n items: 256 threads on
// small systems (latency), 1024 beyond 2 workgroups of 256 per CU so that
// CG_MAXBLK workgroups still fill every wavefront slot.
struct CgGrid {
  int tpb, blocks;
};
static CgGrid cg_grid(int64_t n) {
  CgGrid g;
  g.tpb = n > (int64_t)CG_MAXBLK * 256 ? 1024 : 256;
  g.blocks = (int)std::max<int64_t>(1, std::min<int64_t>((n + g.tpb - 1) / g.tpb, CG_MAXBLK));
  return g;
}

// Scalars of the next direction from state A and the update's partials (slots
// 0 and 1): stop test, beta; the new state in B (first workgroup).  Returns
// false when the iteration has stopped and p must not change; *upd: p is to be
// updated with *beta.  FCG: beta = -(z.q)/(p.q) and the tests of the mixed
// solver's FP32 iteration; else beta = (r.z)/rho and the reference's tests.
// (Fields are read and written one by one: a struct copy per thread is kept
// in memory by the compiler and cost 14 us a launch at 350k equations.)
template <bool FCG>
__device__ inline bool next_direction(const SolveScalars *A, SolveScalars *B, const double *partials, int n0,
                                      int n1, double *beta, bool *upd) {
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  int done = A->done;
  const int pend = A->pend;
  double bt = A->beta, rho = A->rho, resid = A->resid;
  int64_t iter = A->iter;
  if (!done && (pend & 3)) {
    const int slot[2] = {0, 1}, cnt[2] = {pend & 1 ? n0 : 0, pend & 2 ? n1 : 0};
    double t[2];
    sum_slots<2>(partials, slot, cnt, t);
    if (pend & 1) {
      iter++;
      resid = sqrt(t[0]) / A->normb;
      if (FCG) {
        // divergence guard: leave the loop, the host restarts from the true residual
        if (!(resid == resid) || resid > 1e3) done = 3;
        else if (sqrt(t[0]) < A->delta * A->rlast) done = 4;
        else if (iter >= A->maxit) done = 2;
      } else {
        if (resid <= A->tol) done = 1;
        else if (iter >= A->maxit) done = 2;
      }
    }
    if (pend & 2) {
      if (FCG) {
        bt = -t[1] / A->pq;
      } else {
        bt = t[1] / rho;
        rho = t[1];
      }
    }
  } else if (done) {
    if (first) {
      B->done = done;
      B->pend = pend;
      B->iter = iter;
      B->resid = resid;
      B->rho = rho;
      B->beta = bt;
      B->pq = A->pq;
    }
    return false;
  }
  if (first) {
    B->done = done;
    B->pend = 0;
    B->iter = iter;
    B->resid = resid;
    B->rho = rho;
    B->beta = bt;
    B->pq = A->pq;
  }
  *beta = bt;
  *upd = pend != 0;
  // an update request (4) of the FCG still completes its direction
  return !done || (FCG && done == 4);
}

// the update's side of the exchange: state A after a step that ran (pend = 3)
// or after one that found the iteration stopped
__device__ inline void close_step(SolveScalars *A, const SolveScalars *B, double pq, int pend) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    A->iter = B->iter;
    A->resid = B->resid;
    A->rho = B->rho;
    A->beta = B->beta;
    A->pq = pq;
    A->pend = pend;
    A->done = B->done;
  }
}

// end of a batch: the pending test and beta into A (one block), for the host
// and the next batch's first direction
template <bool FCG>
__global__ __launch_bounds__(TPB) void k_cg_close(SolveScalars *A, SolveScalars *B, const double *partials, int n0,
                                                  int n1) {
  double beta;
  bool upd;
  if (A->done || A->pend == 0) return;
  (void)next_direction<FCG>(A, B, partials, n0, n1, &beta, &upd);
  __syncthreads();
  close_step(A, B, B->pq, 4);
}

// PCG64 with the direction formed inside the product: p = z + beta p_old,
// q = K p, partials of p.q (slot 2).  Every gather reads z and p_old and forms
// its entry; the row's own entries go to p_new.
template <int BS>
__global__ __launch_bounds__(TPB) void k_pcg_step64(int64_t nb, const int64_t *__restrict__ bia,
                                                    const int32_t *__restrict__ bja,
                                                    const double *__restrict__ v,
                                                    const double *__restrict__ z,
                                                    const double *__restrict__ p_old,
                                                    double *__restrict__ p_new, double *__restrict__ q,
                                                    const SolveScalars *A, SolveScalars *B, double *partials,
                                                    int n0, int n1) {
  double beta;
  bool upd;
  if (!next_direction<false>(A, B, partials, n0, n1, &beta, &upd)) return;
  const int sub = threadIdx.x % BSR_L;
  constexpr int RPB = TPB / BSR_L;
  double acc = 0.;
  auto dir = [=](int64_t i) { return upd ? beta * p_old[i] + z[i] : p_old[i]; };
  for (int64_t R = (int64_t)blockIdx.x * RPB + threadIdx.x / BSR_L; R < nb; R += (int64_t)gridDim.x * RPB) {
    double out[BS];
    bsr_row_f<double, BS>(R, bia, bja, v, dir, sub, out);
    if (sub < BS) {
      const int64_t i = R * BS + sub;
      const double qi = pick<double, BS>(out, sub), pi = dir(i);
      q[i] = qi;
      p_new[i] = pi;
      acc += qi * pi;
    }
  }
  double vv[1] = {acc};
  store_slots<1>(vv, partials + 2 * MAXBLK);
}

// PCG64 direction alone: p = z + beta p
__global__ __launch_bounds__(1024) void k_pcg_dir64(int64_t n, const double *__restrict__ z,
                                                    double *__restrict__ p, const SolveScalars *A,
                                                    SolveScalars *B, const double *partials, int n0, int n1) {
  double beta;
  bool upd;
  if (!next_direction<false>(A, B, partials, n0, n1, &beta, &upd) || !upd) return;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = beta * p[i] + z[i];
}

// PCG64: q = K p and per-block partial sums of p.q (slot 0)
template <int BS>
__global__ __launch_bounds__(TPB) void k_spmv64_pq(int64_t nb, const int64_t *__restrict__ bia,
                                                   const int32_t *__restrict__ bja,
                                                   const double *__restrict__ v,
                                                   const double *__restrict__ p,
                                                   double *__restrict__ q, const SolveScalars *sc,
                                                   double *partials) {
  if (sc->done) return;
  const int sub = threadIdx.x % BSR_L;
  int64_t lo, hi;
  int xi, xg;
  constexpr int RPB = TPB / BSR_L;  // rows per workgroup tile
#if PZG_XCD_INTERLEAVE
  xcd_slab(nb, lo, hi, xi, xg);
  const int64_t first = lo + (int64_t)xi * RPB, step = (int64_t)xg * RPB;
#else
  xcd_block_range(nb, lo, hi);
  xi = xg = 0;
  const int64_t first = lo, step = RPB;
#endif
  double acc = 0.;
  for (int64_t A = first + threadIdx.x / BSR_L; A < hi; A += step) {
    double out[BS];
    bsr_row<double, BS>(A, bia, bja, v, p, sub, out);
    if (sub < BS) {
      const int64_t i = A * BS + sub;
      const double qi = pick<double, BS>(out, sub);
      q[i] = qi;
      acc += qi * p[i];
    }
  }
  double vv[1] = {acc};
  block_partials<1>(vv, partials);
}

static int bsr_grid(int64_t nb) {
  int64_t g = (nb + TPB / BSR_L - 1) / (TPB / BSR_L);
  if (g > MAXBLK) g = MAXBLK;
  return (int)std::max<int64_t>(g, 1);
}

// x += alpha p; r -= alpha q; partials of r.r (slot 0); preconditioner PRE: 0
// point Jacobi z = r / diag, 1 the connect blocks z = Binv r (BS equations
// each; TPZBlockDiagonal with ELU blocks, the preconditioner
// TPZAnalysis::BuildPreconditioner(EBlockJacobi, true) returns,
// Analysis/TPZAnalysis.cpp:1062-1070), both with r.z in slot 1; 2 left to
// k_vbj_apply64.  alpha = rho / (p.q) from the product's partials (slot 2).
template <int BS, int PRE>
__global__ __launch_bounds__(1024) void k_cg_update64(int64_t nb, double *__restrict__ x,
                                                      double *__restrict__ r,
                                                      double *__restrict__ z,
                                                      const double *__restrict__ p,
                                                      const double *__restrict__ q,
                                                      const double *__restrict__ pre,
                                                      SolveScalars *A, const SolveScalars *B,
                                                      double *partials, int npq) {
  if (B->done) {
    close_step(A, B, B->pq, 0);
    return;
  }
  const int slot[1] = {2}, cnt[1] = {npq};
  double pq[1];
  sum_slots<1>(partials, slot, cnt, pq);
  const double alpha = B->rho / pq[0];
  double rr = 0., rz = 0.;
  for (int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; R < nb; R += (int64_t)gridDim.x * blockDim.x) {
    double rv[BS];
#pragma unroll
    for (int k = 0; k < BS; k++) {
      const int64_t i = R * BS + k;
      x[i] += alpha * p[i];
      rv[k] = r[i] + (-alpha) * q[i];
      r[i] = rv[k];
      rr += rv[k] * rv[k];
    }
    if (PRE == 0) {
#pragma unroll
      for (int k = 0; k < BS; k++) {
        const int64_t i = R * BS + k;
        const double zi = rv[k] / pre[i];
        z[i] = zi;
        rz += rv[k] * zi;
      }
    } else if (PRE == 1) {
      const double *bi = pre + R * BS * BS;
#pragma unroll
      for (int k = 0; k < BS; k++) {
        double t = 0.;
#pragma unroll
        for (int l = 0; l < BS; l++) t += bi[k * BS + l] * rv[l];
        z[R * BS + k] = t;
        rz += rv[k] * t;
      }
    }
  }
  if (PRE == 2) {
    double v[1] = {rr};
    store_slots<1>(v, partials);
  } else {
    double v[2] = {rr, rz};
    store_slots<2>(v, partials);
  }
  close_step(A, B, pq[0], 3);
}

// Connect-block Jacobi of the first residual: p = z = Binv r per block row,
// r.z into partials slot 1.
template <int BS>
__global__ __launch_bounds__(TPB) void k_bj_apply64(int64_t nb, const double *__restrict__ binv,
                                                    const double *__restrict__ r, double *__restrict__ z,
                                                    double *__restrict__ p, double *partials) {
  double rz = 0.;
  for (int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; A < nb; A += (int64_t)gridDim.x * blockDim.x) {
    double rv[BS];
#pragma unroll
    for (int k = 0; k < BS; k++) rv[k] = r[A * BS + k];
    const double *bi = binv + A * BS * BS;
#pragma unroll
    for (int k = 0; k < BS; k++) {
      double s = 0.;
#pragma unroll
      for (int l = 0; l < BS; l++) s += bi[k * BS + l] * rv[l];
      z[A * BS + k] = s;
      p[A * BS + k] = s;
      rz += rv[k] * s;
    }
  }
  __shared__ double sm[TPB / 64];
  const double t = block_sum(rz, sm);
  if (threadIdx.x == 0) partials[1 * MAXBLK + blockIdx.x] = t;
}

// rho = r.z from slot 1 after the block apply of the initial residual
__global__ void k_bj_rho64(SolveScalars *sc, const double *partials, int nblk) {
  const double rz = sum_partials(partials, 1, nblk);
  if (threadIdx.x == 0) sc->rho = rz;
}

// inverse of each diagonal block of K (the first entries of the block's rows
// in the upper CSR; cofactors for 3 x 3, the reciprocal for 1 x 1); a singular
// block sets *fail
template <int BS>
__global__ void k_bj_inv64(int64_t nb, const int64_t *__restrict__ ia, const double *__restrict__ v,
                           double *__restrict__ binv, int *fail) {
  const int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (A >= nb) return;
  double a[BS * BS];
#pragma unroll
  for (int k = 0; k < BS; k++) {
    const int64_t q = ia[A * BS + k];
#pragma unroll
    for (int l = k; l < BS; l++) a[k * BS + l] = a[l * BS + k] = v[q + (l - k)];
  }
  static_assert(BS == 1 || BS == 3, "connect blocks of 1 or 3 equations");
  double *o = binv + A * BS * BS;
  if constexpr (BS == 1) {
    if (a[0] == 0.) atomicExch(fail, 1);
    o[0] = 1. / a[0];
  } else {
    const double c00 = a[4] * a[8] - a[5] * a[7], c01 = a[5] * a[6] - a[3] * a[8], c02 = a[3] * a[7] - a[4] * a[6];
    const double det = a[0] * c00 + a[1] * c01 + a[2] * c02;
    if (det == 0.) atomicExch(fail, 1);
    const double id = 1. / det;
    o[0] = c00 * id;
    o[1] = (a[2] * a[7] - a[1] * a[8]) * id;
    o[2] = (a[1] * a[5] - a[2] * a[4]) * id;
    o[3] = c01 * id;
    o[4] = (a[0] * a[8] - a[2] * a[6]) * id;
    o[5] = (a[2] * a[3] - a[0] * a[5]) * id;
    o[6] = c02 * id;
    o[7] = (a[1] * a[6] - a[0] * a[7]) * id;
    o[8] = (a[0] * a[4] - a[1] * a[3]) * id;
  }
}

// Connect-block Jacobi on high-order meshes: a connect of several shapes
// is one block of its consecutive equations [pos, pos + m), m <= VBJ_MAX.
// Inverse: one wavefront per block, the block (from the upper CSR, whose
// row i starts with the columns i, i+1, ... of its own connect) and the
// identity in LDS, Gauss-Jordan with lane r holding row r; a missing entry
// or a zero pivot sets *fail.
__global__ __launch_bounds__(256) void k_vbj_inv64(int64_t nblk, const int64_t *__restrict__ bpos,
                                                   const int32_t *__restrict__ bm,
                                                   const int64_t *__restrict__ boff,
                                                   const int64_t *__restrict__ ia,
                                                   const int64_t *__restrict__ ja,
                                                   const double *__restrict__ a, double *__restrict__ binv,
                                                   int *fail) {
  __shared__ double sA[4][VBJ_MAX][VBJ_MAX], sI[4][VBJ_MAX][VBJ_MAX];
  const int w = threadIdx.x >> 6, r = threadIdx.x & 63;
  const int64_t b = (int64_t)blockIdx.x * 4 + w;
  if (b >= nblk) return;  // whole wavefronts
  const int64_t p = bpos[b];
  const int m = bm[b];
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  if (r < m)
    for (int c = 0; c < m; c++) {
      const int lo = r < c ? r : c, hi = r < c ? c : r;
      const int64_t q = ia[p + lo] + (hi - lo);
      if (q >= ia[p + lo + 1] || ja[q] != p + hi) atomicExch(fail, 1);
      sA[w][r][c] = q < ia[p + lo + 1] ? a[q] : 0.;
      sI[w][r][c] = r == c ? 1. : 0.;
    }
  sync();
  for (int k = 0; k < m; k++) {
    const double piv = sA[w][k][k];
    if (piv == 0.) {
      if (r == 0) atomicExch(fail, 1);
      return;
    }
    sync();
    if (r == k)
      for (int c = 0; c < m; c++) {
        sA[w][k][c] /= piv;
        sI[w][k][c] /= piv;
      }
    sync();
    if (r < m && r != k) {
      const double f = sA[w][r][k];
      for (int c = 0; c < m; c++) {
        sA[w][r][c] -= f * sA[w][k][c];
        sI[w][r][c] -= f * sI[w][k][c];
      }
    }
    sync();
  }
  if (r < m)
    for (int c = 0; c < m; c++) binv[boff[b] + (int64_t)r * m + c] = sI[w][r][c];
}

// z = Binv r on the blocks (one thread per equation), r.z into partials
// slot 1; p = z too when p is given (the first residual)
__global__ __launch_bounds__(TPB) void k_vbj_apply64(int64_t n, const int32_t *__restrict__ eqb,
                                                     const int64_t *__restrict__ bpos,
                                                     const int32_t *__restrict__ bm,
                                                     const int64_t *__restrict__ boff,
                                                     const double *__restrict__ binv,
                                                     const double *__restrict__ r, double *__restrict__ z,
                                                     double *__restrict__ p, const SolveScalars *sc,
                                                     double *partials) {
  if (sc && sc->done) return;
  double rz = 0.;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t b = eqb[i];
    const int64_t b0 = bpos[b];
    const int m = bm[b];
    const double *row = binv + boff[b] + (i - b0) * m;
    double s = 0.;
    for (int c = 0; c < m; c++) s += row[c] * r[b0 + c];
    z[i] = s;
    if (p) p[i] = s;
    rz += r[i] * s;
  }
  __shared__ double sm[TPB / 64];
  const double t = block_sum(rz, sm);
  if (threadIdx.x == 0) partials[1 * MAXBLK + blockIdx.x] = t;
}

// The connect blocks of the scaled FP32 operator S = D^-1/2 K D^-1/2:
// S_b^-1 = D^1/2 K_b^-1 D^1/2, from the FP64 inverses (one thread per row)
__global__ void k_vbj_scale32(int64_t n, const int32_t *__restrict__ eqb, const int64_t *__restrict__ bpos,
                              const int32_t *__restrict__ bm, const int64_t *__restrict__ boff,
                              const double *__restrict__ inv64, const double *__restrict__ dis,
                              float *__restrict__ inv32) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t b = eqb[i];
    const int64_t p = bpos[b], o = boff[b] + (i - p) * bm[b];
    for (int c = 0; c < bm[b]; c++) inv32[o + c] = (float)(inv64[o + c] / (dis[i] * dis[p + c]));
  }
}

// FP32 FCG with the connect blocks: z = S_b^-1 r (one thread per equation);
// p = z at a restart; z.q replaces slot 1 of the FCG update's partials
// (launched on the same grid)
__global__ __launch_bounds__(TPB) void k_vbj_apply32(int64_t n, const int32_t *__restrict__ eqb,
                                                     const int64_t *__restrict__ bpos,
                                                     const int32_t *__restrict__ bm,
                                                     const int64_t *__restrict__ boff,
                                                     const float *__restrict__ inv, const float *__restrict__ r,
                                                     float *__restrict__ z, float *__restrict__ p,
                                                     const float *__restrict__ q, const SolveScalars *sc,
                                                     double *partials) {
  if (sc && sc->done) return;
  double zq = 0.;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t b = eqb[i];
    const int64_t s0 = bpos[b];
    const int m = bm[b];
    const float *row = inv + boff[b] + (i - s0) * m;
    float v = 0.f;
    for (int c = 0; c < m; c++) v += row[c] * r[s0 + c];
    z[i] = v;
    if (p) p[i] = v;
    if (q) zq += (double)v * q[i];
  }
  if (!q) return;
  __shared__ double sm[TPB / 64];
  const double t = block_sum(zq, sm);
  if (threadIdx.x == 0) partials[1 * MAXBLK + blockIdx.x] = t;
}

// x = 0; r = b; p = z = r/diag (with diag); rho = r.z; normb = |b|
__global__ __launch_bounds__(TPB) void k_cg_init64(int64_t n, const double *__restrict__ b,
                                                   double *__restrict__ x, double *__restrict__ r,
                                                   double *__restrict__ z, double *__restrict__ p,
                                                   const double *__restrict__ diag,
                                                   SolveScalars *sc, double *partials) {
  double bb = 0., rz = 0.;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    double bi = b[i];
    x[i] = 0.;
    r[i] = bi;
    bb += bi * bi;
    if (diag) {
      double zi = bi / diag[i];
      z[i] = zi;
      p[i] = zi;
      rz += bi * zi;
    }
  }
  double v[2] = {bb, rz};
  block_partials<2>(v, partials);
}
__global__ void k_fin_cg_init64(SolveScalars *sc, const double *partials, int nblk) {
  const double bb = sum_partials(partials, 0, nblk), rz = sum_partials(partials, 1, nblk);
  if (threadIdx.x == 0) {
    double normb = sqrt(bb);
    double resid = normb == 0. ? 0. : 1.0;
    if (normb == 0.) normb = 1.;
    sc->normb = normb;
    sc->resid = resid;
    sc->iter = 0;
    sc->rho = rz;
    sc->beta = 0.;
    sc->done = resid <= sc->tol ? 1 : 0;
  }
}

// Continuation from the current x with its residual r = f - K x already in
// r (CG<> with fromCurrent, Solvers/LinearSolvers/cg.h:29-132): p = z = r/diag,
// rho = r.z, normb = |f|, resid = |r|/|f|.
__global__ __launch_bounds__(TPB) void k_cg_restart64(int64_t n, const double *__restrict__ f,
                                                      const double *__restrict__ r,
                                                      double *__restrict__ z, double *__restrict__ p,
                                                      const double *__restrict__ diag,
                                                      SolveScalars *sc, double *partials) {
  double ff = 0., rr = 0., rz = 0.;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    const double fi = f[i], ri = r[i], zi = ri / diag[i];
    p[i] = zi;
    z[i] = zi;
    ff += fi * fi;
    rr += ri * ri;
    rz += ri * zi;
  }
  double v[3] = {ff, rr, rz};
  block_partials<3>(v, partials);
}
__global__ void k_fin_cg_restart64(SolveScalars *sc, const double *partials, int nblk) {
  const double ff = sum_partials(partials, 0, nblk), rr = sum_partials(partials, 1, nblk),
               rz = sum_partials(partials, 2, nblk);
  if (threadIdx.x == 0) {
    double normb = sqrt(ff);
    if (normb == 0.) normb = 1.;
    const double resid = sqrt(rr) / normb;
    sc->normb = normb;
    sc->resid = resid;
    sc->rho = rz;
    sc->beta = 0.;
    sc->done = resid <= sc->tol ? 1 : 0;
  }
}

// r = f - K u (FP64 block CSR), |r|^2 and |f|^2
template <int BS>
__global__ __launch_bounds__(TPB) void k_residual64(int64_t nb, const int64_t *__restrict__ bia,
                                                    const int32_t *__restrict__ bja,
                                                    const double *__restrict__ v,
                                                    const double *__restrict__ u,
                                                    const double *__restrict__ f,
                                                    double *__restrict__ r, double *partials) {
  const int sub = threadIdx.x % BSR_L;
  int64_t lo, hi;
  int xi, xg;
  constexpr int RPB = TPB / BSR_L;  // rows per workgroup tile
#if PZG_XCD_INTERLEAVE
  xcd_slab(nb, lo, hi, xi, xg);
  const int64_t first = lo + (int64_t)xi * RPB, step = (int64_t)xg * RPB;
#else
  xcd_block_range(nb, lo, hi);
  xi = xg = 0;
  const int64_t first = lo, step = RPB;
#endif
  double rr = 0., ff = 0.;
  for (int64_t A = first + threadIdx.x / BSR_L; A < hi; A += step) {
    double o[BS];
    bsr_row<double, BS>(A, bia, bja, v, u, sub, o);
    if (sub < BS) {
      const int64_t i = A * BS + sub;
      const double ri = f[i] - pick<double, BS>(o, sub);
      if (r) r[i] = ri;
      rr += ri * ri;
      ff += f[i] * f[i];
    }
  }
  double vv[2] = {rr, ff};
  block_partials<2>(vv, partials);
}
// out = (|r|^2, |f|^2) from the residual's partials (one block; |r|^2 twice
// when only slot 0 was written)
__global__ void k_fin_residual64(const double *partials, int nblk, int nslot, double *out) {
  const double rr = sum_partials(partials, 0, nblk);
  const double ff = nslot > 1 ? sum_partials(partials, 1, nblk) : rr;
  if (threadIdx.x == 0) {
    out[0] = rr;
    out[1] = ff;
  }
}

// the residual of u = 0: r = f, out = (|f|^2, |f|^2)
__global__ __launch_bounds__(TPB) void k_residual_zero(int64_t n, const double *__restrict__ f,
                                                       double *__restrict__ r, double *partials) {
  double ff = 0.;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double v = f[i];
    r[i] = v;
    ff += v * v;
  }
  double vv[1] = {ff};
  block_partials<1>(vv, partials);
}

// ---- small systems: CG in one workgroup ------------------------------------
// The whole iteration of a system whose block CSR and vectors fit in one CU's
// LDS runs in one workgroup: matrix, p, q, r, x and the preconditioner in LDS,
// three barriers an iteration, no launch in between.  Bound by LDS latency:
// 3.2 us an iteration at 289 equations (Poisson 8^2 p = 2, solve 0.27 ms
// against 3.3 ms of launches).  A launch runs at most CG_SMALL_IT iterations and
// leaves its state (x, r, p, scalars) in memory, where the next one resumes.
constexpr int CG_SMALL_TPB = 1024;
constexpr int CG_SMALL_IT = 2000;
constexpr int64_t CG_SMALL_LDS = 158 * 1024;  // of the CU's 160 KB; the rest is the reductions'

template <int BS>
static int64_t cg_small_lds(int64_t nb, int64_t nbf, bool block) {
  const int64_t n = nb * BS;
  return 8 * (nbf * BS * BS + n * (4 + (block ? BS : 1))) + 4 * (nbf + nb + 1);
}

// L lanes (a power of two <= 16) per scalar row in the product; vector steps
// one thread per block row.
template <int BS, bool BLOCK>
__global__ __launch_bounds__(CG_SMALL_TPB) void k_cg_small(int nb, int nbf, int L,
                                                           const int64_t *__restrict__ bia,
                                                           const int32_t *__restrict__ bja,
                                                           const double *__restrict__ v,
                                                           const double *__restrict__ pre,
                                                           double *__restrict__ xg, double *__restrict__ rg,
                                                           double *__restrict__ pg, SolveScalars *sc) {
  constexpr int BB = BS * BS;
  extern __shared__ double lds[];
  __shared__ double sm[3][CG_SMALL_TPB / 64];
  if (sc->done) return;
  const int n = nb * BS, tid = threadIdx.x, w = tid >> 6;
  double *sv = lds, *p = sv + (int64_t)nbf * BB, *q = p + n, *r = q + n, *x = r + n, *m = x + n;
  int32_t *cj = reinterpret_cast<int32_t *>(m + (int64_t)n * (BLOCK ? BS : 1)), *ci = cj + nbf;
  for (int i = tid; i < nbf * BB; i += CG_SMALL_TPB) sv[i] = v[i];
  for (int i = tid; i < nbf; i += CG_SMALL_TPB) cj[i] = bja[i];
  for (int i = tid; i <= nb; i += CG_SMALL_TPB) ci[i] = (int32_t)bia[i];
  for (int i = tid; i < n; i += CG_SMALL_TPB) {
    p[i] = pg[i];
    r[i] = rg[i];
    x[i] = xg[i];
  }
  for (int i = tid; i < n * (BLOCK ? BS : 1); i += CG_SMALL_TPB) m[i] = pre[i];
  // total of one value per thread in every thread (slot k of sm; a slot is
  // written again only after another barrier)
  auto total = [&](double s, int k) {
    s = wave_sum(s);
    if ((tid & 63) == 0) sm[k][w] = s;
  };
  auto read = [&](int k) {
    double t = 0.;
    for (int j = 0; j < CG_SMALL_TPB / 64; j++) t += sm[k][j];
    return t;
  };
  const double normb = sc->normb, tol = sc->tol;
  double rho = sc->rho, beta = sc->beta, resid = sc->resid;
  int64_t it = sc->iter;
  const int64_t maxit = sc->maxit;
  int done = 0;
  const int sub = tid & (L - 1), grp = tid / L, ngrp = CG_SMALL_TPB / L;
  __syncthreads();
  for (int k = 0; k < CG_SMALL_IT && !done; k++) {
    double pq = 0.;
    for (int i0 = 0; i0 < n; i0 += ngrp) {  // every lane of a wavefront runs the same passes
      const int i = i0 + grp, A = i / BS, c = i - A * BS;
      double s = 0.;
      if (i < n) {
        const int b0 = ci[A], nn = ci[A + 1] - b0;
        for (int j = sub; j < nn; j += L) {
          const int j0 = BS == 1 ? j : j / BSR_CHUNK * BSR_CHUNK;
          const int mc = BS == 1 ? 1 : (nn - j0 < BSR_CHUNK ? nn - j0 : BSR_CHUNK);
          const double *vp = sv + (b0 + j0) * BB + (j - j0);
          const double *pp = p + cj[b0 + j] * BS;
#pragma unroll
          for (int l = 0; l < BS; l++) s += vp[(c * BS + l) * mc] * pp[l];
        }
      }
      for (int o = L >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (i < n && sub == 0) {
        q[i] = s;
        pq += s * p[i];
      }
    }
    total(pq, 0);
    __syncthreads();
    const double alpha = rho / read(0);
    double rr = 0., rz = 0.;
    for (int A = tid; A < nb; A += CG_SMALL_TPB) {
      double rv[BS];
#pragma unroll
      for (int a = 0; a < BS; a++) {
        const int i = A * BS + a;
        x[i] += alpha * p[i];
        rv[a] = r[i] + (-alpha) * q[i];
        r[i] = rv[a];
        rr += rv[a] * rv[a];
      }
#pragma unroll
      for (int a = 0; a < BS; a++) {
        const int i = A * BS + a;
        double z = 0.;
        if (BLOCK) {
#pragma unroll
          for (int l = 0; l < BS; l++) z += m[(A * BS + a) * BS + l] * rv[l];
        } else {
          z = rv[a] / m[i];
        }
        q[i] = z;
        rz += rv[a] * z;
      }
    }
    total(rr, 1);
    total(rz, 2);
    __syncthreads();
    it++;
    resid = sqrt(read(1)) / normb;
    if (resid <= tol) done = 1;
    else if (it >= maxit) done = 2;
    const double t = read(2);
    beta = t / rho;
    rho = t;
    if (!done)
      for (int A = tid; A < nb; A += CG_SMALL_TPB)
#pragma unroll
        for (int a = 0; a < BS; a++) p[A * BS + a] = beta * p[A * BS + a] + q[A * BS + a];
    __syncthreads();
  }
  for (int i = tid; i < n; i += CG_SMALL_TPB) {
    pg[i] = p[i];
    rg[i] = r[i];
    xg[i] = x[i];
  }
  if (tid == 0) {
    sc->iter = it;
    sc->resid = resid;
    sc->beta = beta;
    sc->rho = rho;
    sc->pend = 0;
    sc->done = done;
  }
}

__global__ void k_axpby64(int64_t n, double alpha, const double *__restrict__ x, double beta,
                          const double *__restrict__ y, double *__restrict__ z) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) z[i] = alpha * x[i] + (y ? beta * y[i] : 0.);
}

#define DISPATCH_BS(BSV, CALL)                         \
  switch (BSV) {                                       \
    case 3: { constexpr int BS = 3; CALL; } break;     \
    default: { constexpr int BS = 1; CALL; } break;    \
  }

int launch_spmv64(Ctx &c, const double *x, double *y) {
  DISPATCH_BS(c.bs, hipLaunchKernelGGL((k_spmv_bsr<double, BS>), dim3(bsr_grid(c.nb)), dim3(TPB), 0,
                                       c.stream, c.nb, c.d_fbia.as<int64_t>(),
                                       c.d_fbja.as<int32_t>(), c.d_fa.as<double>(), x, y));
  PZG_HIP(hipGetLastError());
  return PZG_OK;
}

static int ensure_reduce(Ctx &c) {
  if (!c.d_partials.p) {
    PZG_TRY(dev_alloc(c.d_partials, sizeof(double) * NSLOT * MAXBLK));
    PZG_TRY(dev_alloc(c.d_flag, sizeof(int)));
  }
  PZG_TRY(dev_alloc(c.d_scal, sizeof(SolveScalars) * 2));
  PZG_TRY(dev_alloc(c.d_res2, 2 * sizeof(double)));
  return PZG_OK;
}
int ensure_reduce_pub(Ctx &c) { return ensure_reduce(c); }

static void fin_residual64(Ctx &c, const double *partials, int nblk, int nslot, double *out) {
  hipLaunchKernelGGL(k_fin_residual64, dim3(1), dim3(TPB), 0, c.stream, partials, nblk, nslot, out);
}

int launch_multadd_upper(Ctx &c, const double *x, const double *y, double *z, double alpha,
                         double beta) {
  bool kf = false;
  PZG_TRY(kf_prepare(c, &kf));
  if (kf) return kf_apply(c, KF_AXPBY, x, y, alpha, beta, z, nullptr, nullptr);
  if (!c.full_valid) PZG_TRY(launch_expand_full(c));
  PZG_TRY(launch_spmv64(c, x, z));
  int64_t n = c.neq;
  hipLaunchKernelGGL(k_axpby64, dim3(grid_for(n, TPB)), dim3(TPB), 0, c.stream, n, alpha, z, beta,
                     y, z);
  PZG_HIP(hipGetLastError());
  return PZG_OK;
}

// r = f - K u (r may be null) and out = (|r|^2, |f|^2), by the element
// products when they are prepared (kf_prepare) and the block CSR otherwise
static int launch_residual64(Ctx &c, const double *u, double *r, double *partials, double *out) {
  if (c.kf_valid) {
    PZG_TRY(kf_apply(c, KF_RESIDUAL, u, c.d_f.as<double>(), 1., 0., r, nullptr, partials));
    fin_residual64(c, partials, kf_rows_grid(c), 2, out);
  } else {
    DISPATCH_BS(c.bs, hipLaunchKernelGGL(k_residual64<BS>, dim3(bsr_grid(c.nb)), dim3(TPB), 0, c.stream, c.nb,
                                         c.d_fbia.as<int64_t>(), c.d_fbja.as<int32_t>(), c.d_fa.as<double>(), u,
                                         c.d_f.as<double>(), r, partials));
    fin_residual64(c, partials, bsr_grid(c.nb), 2, out);
  }
  PZG_HIP(hipGetLastError());
  return PZG_OK;
}

// the FP64 operator of the assembled system: element products or block CSR
static int prepare_k64(Ctx &c) {
  bool kf = false;
  PZG_TRY(kf_prepare(c, &kf));
  if (!kf && !c.full_valid) PZG_TRY(launch_expand_full(c));
  return PZG_OK;
}

int true_residual(Ctx &c, const double *u, double *rel) {
  if (!c.f_valid || !c.d_f.p || !u) {  // never launch on a missing load or solution
    set_error("true residual: no load or solution of the current system on the device");
    return PZG_ESTATE;
  }
  PZG_TRY(prepare_k64(c));
  PZG_TRY(ensure_reduce(c));
  PZG_TRY(launch_residual64(c, u, nullptr, c.d_partials.as<double>(), c.d_res2.as<double>()));
  double h[2];
  PZG_HIP(hipMemcpyAsync(h, c.d_res2.p, sizeof(h), hipMemcpyDeviceToHost, c.stream));
  PZG_HIP(hipStreamSynchronize(c.stream));
  *rel = h[1] > 0 ? std::sqrt(h[0] / h[1]) : std::sqrt(h[0]);
  return PZG_OK;
}

// ---- allocation-free true residual ---------------------------------------
// Fixed device scratch of pzg_true_residual_noalloc, one copy per GPU, held
// until the process ends: the reduction partials (2 x MAXBLK doubles, one slot
// per workgroup of the capped residual grid) and the two sums.  32.8 KB
// whatever the system size: the residual kernels stride over the rows with at
// most MAXBLK workgroups.
constexpr int NOALLOC_PART = 2 * MAXBLK;           // partials, doubles
constexpr int NOALLOC_OUT = NOALLOC_PART;          // |r|^2, |f|^2
constexpr int NOALLOC_WORDS = NOALLOC_PART + 2;
static __device__ __align__(256) double scratch[NOALLOC_WORDS];

constexpr int NOALLOC_MAXDEV = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[NOALLOC_MAXDEV] = {};

// Looks up this device's address of 'scratch' (the host-side name is only a
// stand-in).  Called by pzg_create with the context's device current.
int noalloc_scratch_setup(int device) {
  if (device < 0 || device >= NOALLOC_MAXDEV) {
    set_error("pzg_create: device index beyond the allocation-free scratch table");
    return PZG_EINVAL;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return PZG_OK;
  void *p = nullptr;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    return PZG_EHIP;
  }
  g_scratch_ptr[device] = static_cast<double *>(p);
  return PZG_OK;
}

// The residual of true_residual on the FP64 operator already on the device
// (element products or full block CSR), reducing in the per-device scratch: no
// allocation of any kind.
int true_residual_noalloc(Ctx &c, double *rel) {
  if (!(c.kf_valid || (c.full_valid && c.d_fbia.p)) || !c.f_valid || !c.d_f.p) {
    set_error("pzg_true_residual_noalloc: no FP64 operator or load of the current system on the "
              "device (call a solve or pzg_true_residual after assembling first)");
    return PZG_ESTATE;
  }
  double *s = (c.device >= 0 && c.device < NOALLOC_MAXDEV) ? g_scratch_ptr[c.device] : nullptr;
  if (!s) {
    set_error("pzg_true_residual_noalloc: scratch of this device not set up");
    return PZG_ESTATE;
  }
  const int grid = c.kf_valid ? kf_rows_grid(c) : bsr_grid(c.nb);
  if (grid > NOALLOC_PART / 2) {
    set_error("pzg_true_residual_noalloc: residual grid of " + std::to_string(grid) +
              " workgroups exceeds the scratch's " + std::to_string(NOALLOC_PART / 2));
    return PZG_EINVAL;
  }
  PZG_TRY(launch_residual64(c, c.d_u.as<double>(), nullptr, s, s + NOALLOC_OUT));
  double h[2];
  PZG_HIP(hipMemcpyAsync(h, s + NOALLOC_OUT, sizeof(h), hipMemcpyDeviceToHost, c.stream));
  PZG_HIP(hipStreamSynchronize(c.stream));
  *rel = h[1] > 0 ? std::sqrt(h[0] / h[1]) : std::sqrt(h[0]);
  return PZG_OK;
}

// Runs batches of the given enqueue function, optionally through a captured
// hipGraph, until the device 'done' flag is set.  key: everything the captured
// launches hold (pointers, sizes, launch shapes); the context keeps the last
// graph and reuses it while the key is the same (capture and instantiation of
// 100 iterations cost 0.5 to 1.5 ms a solve).  An empty key: used here only.
template <class F>
static int run_batches(Ctx &c, bool use_graph, std::vector<uint64_t> key, F enqueue, SolveScalars &hs) {
  hipGraphExec_t exec = nullptr;
  const bool keep = !key.empty();
  if (use_graph && keep && c.solve_graph && c.solve_key == key) exec = c.solve_graph;
  if (use_graph && !exec) {
    hipGraph_t graph = nullptr;
    PZG_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
    enqueue();
    PZG_HIP(hipStreamEndCapture(c.stream, &graph));
    const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
      set_error(std::string("pzg_solve: hipGraphInstantiate: ") + hipGetErrorString(e));
      return PZG_EHIP;
    }
    if (keep) {
      if (c.solve_graph) (void)hipGraphExecDestroy(c.solve_graph);
      c.solve_graph = exec;
      c.solve_key.swap(key);
    }
  }
  int rc = PZG_OK;
  for (;;) {
    hipError_t e = hipSuccess;
    if (use_graph) e = hipGraphLaunch(exec, c.stream);
    else enqueue();
    if (e == hipSuccess) e = hipMemcpyAsync(&hs, c.d_scal.p, sizeof(SolveScalars), hipMemcpyDeviceToHost, c.stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
    if (e != hipSuccess) {
      set_error(std::string("pzg_solve: iteration batch: ") + hipGetErrorString(e));
      rc = PZG_EHIP;
      break;
    }
    if (hs.done) break;
  }
  if (exec && !keep) (void)hipGraphExecDestroy(exec);
  return rc;
}

// q = K p with the partials of p.q in slot 2; the number of partials
static int pq64_grid(const Ctx &c) { return c.kf_valid ? kf_rows_grid(c) : bsr_grid(c.nb); }
static void launch_pq64(Ctx &c, SolveScalars *sc, double *part) {
  if (c.kf_valid) {
    (void)kf_apply(c, KF_DOT, c.d_p.as<double>(), nullptr, 1., 0., c.d_q.as<double>(), sc, part + 2 * MAXBLK);
    return;
  }
  DISPATCH_BS(c.bs, hipLaunchKernelGGL(k_spmv64_pq<BS>, dim3(bsr_grid(c.nb)), dim3(TPB), 0, c.stream, c.nb,
                                       c.d_fbia.as<int64_t>(), c.d_fbja.as<int32_t>(), c.d_fa.as<double>(),
                                       c.d_p.as<double>(), c.d_q.as<double>(), sc, part + 2 * MAXBLK));
}

enum { PRE_JACOBI = 0, PRE_BLOCK = 1, PRE_VBLOCK = 2 };
// Direction formed inside the product (two launches an iteration) up to this
// many stored scalars, beyond as a launch of its own: the second gathered
// vector costs more than the launch once the product is bound by its gathers.
// Merged against apart, ms per solve: 263k scalars (Poisson 64^2 p = 2) 2.99 /
// 3.29, 456k (elasticity 12^3 p = 1) 6.81 / 6.91, 920k (Poisson 120^2) 9.63 /
// 7.78; FCG: 0.4M (elasticity hp 8^3) 8.42 / 8.57, 6M (hp 21^3) 29.0 / 25.9,
// 21M (tetrahedra, orders to 5) 109 / 34.
constexpr int64_t PCG_MERGE_NNZ = (int64_t)1 << 19;

// Iterations of PCG64 from the state that the start kernels left (x = d_u,
// r = d_r, p = z, scalars in d_scal) until tol, maxit; hs receives the scalars.
template <int BS>
static int pcg64_iterate(Ctx &c, const pzg_solve_params &prm, int pre, SolveScalars &hs) {
  const int64_t n = c.neq, nb = c.nb;
  SolveScalars *A = c.d_scal.as<SolveScalars>(), *B = A + 1;
  double *part = c.d_partials.as<double>();
  const double *m = pre == PRE_JACOBI ? c.d_diag.as<double>() : c.d_bjinv64.as<double>();
  const int64_t lds = cg_small_lds<BS>(nb, c.nbf, pre == PRE_BLOCK);
  if (!c.kf_valid && pre != PRE_VBLOCK && lds <= CG_SMALL_LDS) {
    int L = 1;
    while (L < 16 && n * L * 2 <= CG_SMALL_TPB) L *= 2;
    const void *fn = pre == PRE_BLOCK ? (const void *)k_cg_small<BS, true> : (const void *)k_cg_small<BS, false>;
    PZG_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)CG_SMALL_LDS));
    do {
      if (pre == PRE_BLOCK)
        hipLaunchKernelGGL((k_cg_small<BS, true>), dim3(1), dim3(CG_SMALL_TPB), (size_t)lds, c.stream, (int)nb,
                           (int)c.nbf, L, c.d_fbia.as<int64_t>(), c.d_fbja.as<int32_t>(), c.d_fa.as<double>(), m,
                           c.d_u.as<double>(), c.d_r.as<double>(), c.d_p.as<double>(), A);
      else
        hipLaunchKernelGGL((k_cg_small<BS, false>), dim3(1), dim3(CG_SMALL_TPB), (size_t)lds, c.stream, (int)nb,
                           (int)c.nbf, L, c.d_fbia.as<int64_t>(), c.d_fbja.as<int32_t>(), c.d_fa.as<double>(), m,
                           c.d_u.as<double>(), c.d_r.as<double>(), c.d_p.as<double>(), A);
      PZG_HIP(hipGetLastError());
      PZG_HIP(hipMemcpyAsync(&hs, A, sizeof(hs), hipMemcpyDeviceToHost, c.stream));
      PZG_HIP(hipStreamSynchronize(c.stream));
    } while (!hs.done);
    return PZG_OK;
  }
  const CgGrid gu = cg_grid(nb), gd = cg_grid(n);
  const int gv = grid_for(n, TPB), gs = pq64_grid(c);
  const int n1 = pre == PRE_VBLOCK ? gv : gu.blocks;
  const bool merge = !c.kf_valid && c.nbf * BS * BS <= PCG_MERGE_NNZ;
  if (merge) PZG_TRY(dev_alloc(c.d_p2, n * sizeof(double)));
  const int gm = std::min(gs, CG_MAXBLK);
  double *r = c.d_r.as<double>(), *z = c.d_z.as<double>(), *q = c.d_q.as<double>(), *x = c.d_u.as<double>();
  auto step = [&](double *p_old, double *p_new) {
    double *p = merge ? p_new : c.d_p.as<double>();
    if (merge) {
      hipLaunchKernelGGL(k_pcg_step64<BS>, dim3(gm), dim3(TPB), 0, c.stream, nb, c.d_fbia.as<int64_t>(),
                         c.d_fbja.as<int32_t>(), c.d_fa.as<double>(), (const double *)z, (const double *)p_old, p_new,
                         q, (const SolveScalars *)A, B, part, gu.blocks, n1);
    } else {
      hipLaunchKernelGGL(k_pcg_dir64, dim3(gd.blocks), dim3(gd.tpb), 0, c.stream, n, (const double *)z, p,
                         (const SolveScalars *)A, B, (const double *)part, gu.blocks, n1);
      launch_pq64(c, B, part);
    }
    const int npq = merge ? gm : gs;
#define PZG_UPD(P)                                                                                               \
  hipLaunchKernelGGL((k_cg_update64<BS, P>), dim3(gu.blocks), dim3(gu.tpb), 0, c.stream, nb, x, r, z,            \
                     (const double *)p, (const double *)q, m, A, (const SolveScalars *)B, part, npq)
    if (pre == PRE_JACOBI) PZG_UPD(0);
    else if (pre == PRE_BLOCK) PZG_UPD(1);
    else PZG_UPD(2);
#undef PZG_UPD
    if (pre == PRE_VBLOCK)
      hipLaunchKernelGGL(k_vbj_apply64, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_vbj_eqb.as<int32_t>(),
                         c.d_vbj_pos.as<int64_t>(), c.d_vbj_m.as<int32_t>(), c.d_vbj_off.as<int64_t>(), m,
                         (const double *)r, z, (double *)nullptr, (const SolveScalars *)A, part);
  };
  // an even number of iterations: the two direction buffers are back in place
  const int batch = ((prm.check_every > 0 ? prm.check_every : 50) + 1) / 2 * 2;
  auto enqueue = [&]() {
    double *p0 = c.d_p.as<double>(), *p1 = merge ? c.d_p2.as<double>() : p0;
    for (int k = 0; k < batch; k += 2) {
      step(p0, p1);
      step(p1, p0);
    }
    hipLaunchKernelGGL(k_cg_close<false>, dim3(1), dim3(TPB), 0, c.stream, A, B, (const double *)part, gu.blocks, n1);
  };
  std::vector<uint64_t> key;
  key_add(key, 64, BS, pre, batch, n, nb, c.nbf, merge, c.kf_valid);
  for (const DevBuf *b : {&c.d_scal, &c.d_partials, &c.d_r, &c.d_z, &c.d_q, &c.d_u, &c.d_p, &c.d_p2, &c.d_diag,
                          &c.d_bjinv64, &c.d_fbia, &c.d_fbja, &c.d_fa, &c.d_vbj_eqb, &c.d_vbj_pos, &c.d_vbj_m,
                          &c.d_vbj_off})
    key_add(key, *b);
  if (c.kf_valid) kf_key(c, key);
  return run_batches(c, prm.use_graph != 0, key, enqueue, hs);
}

// FP64 Jacobi-PCG iterations (the EJacobi CG<> of solve_pcg64) continued from
// the current solution u, whose true residual f - K u is in d_r: the mixed
// solver's fallback when the FP32 iterations stall.  Runs until the
// recursive residual reaches 0.9 tol, then checks the true residual; at most
// four such restarts.  iters accumulates the iterations; rel receives the
// true relative residual.
static int pcg64_continue(Ctx &c, const pzg_solve_params &prm, int64_t &iters, double &rel) {
  const int64_t n = c.neq;
  for (DevBuf *b : {&c.d_z, &c.d_p, &c.d_q}) PZG_TRY(dev_alloc(*b, n * sizeof(double)));
  SolveScalars *sc = c.d_scal.as<SolveScalars>();
  double *part = c.d_partials.as<double>();
  const int gv = grid_for(n, TPB);
  for (int round = 0; round < 4 && rel > prm.tol && iters < prm.max_iter; round++) {
    SolveScalars hs;
    std::memset(&hs, 0, sizeof(hs));
    hs.tol = 0.9 * prm.tol;
    hs.maxit = prm.max_iter;
    hs.iter = iters;
    PZG_HIP(hipMemcpyAsync(c.d_scal.p, &hs, sizeof(hs), hipMemcpyHostToDevice, c.stream));
    hipLaunchKernelGGL(k_cg_restart64, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_f.as<double>(),
                       c.d_r.as<double>(), c.d_z.as<double>(), c.d_p.as<double>(),
                       c.d_diag.as<double>(), sc, part);
    hipLaunchKernelGGL(k_fin_cg_restart64, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gv);
    PZG_HIP(hipGetLastError());
    PZG_HIP(hipMemcpyAsync(&hs, c.d_scal.p, sizeof(hs), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    if (!hs.done) {
      int rc = PZG_OK;
      DISPATCH_BS(c.bs, rc = pcg64_iterate<BS>(c, prm, PRE_JACOBI, hs));
      PZG_TRY(rc);
    }
    iters = hs.iter;
    // true residual into d_r (the next round restarts from it)
    PZG_TRY(launch_residual64(c, c.d_u.as<double>(), c.d_r.as<double>(), part, c.d_res2.as<double>()));
    double h[2];
    PZG_HIP(hipMemcpyAsync(h, c.d_res2.p, sizeof(h), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    rel = h[1] > 0 ? std::sqrt(h[0] / h[1]) : std::sqrt(h[0]);
    if (hs.done == 2) break;
  }
  return PZG_OK;
}

int solve_pcg64(Ctx &c, const pzg_solve_params &prm, pzg_solve_info &info) {
  const int64_t n = c.neq;
  PZG_TRY(prepare_k64(c));
  PZG_TRY(ensure_reduce(c));
  for (DevBuf *b : {&c.d_u, &c.d_r, &c.d_z, &c.d_p, &c.d_q}) PZG_TRY(dev_alloc(*b, n * sizeof(double)));
  SolveScalars hs;
  std::memset(&hs, 0, sizeof(hs));
  hs.tol = prm.tol;
  hs.maxit = prm.max_iter;
  PZG_HIP(hipMemcpyAsync(c.d_scal.p, &hs, sizeof(hs), hipMemcpyHostToDevice, c.stream));
  PZG_HIP(hipEventRecord(c.ev0, c.stream));
  SolveScalars *sc = c.d_scal.as<SolveScalars>();
  double *part = c.d_partials.as<double>();
  const int gv = grid_for(n, TPB);
  // EJacobi (reference default) or the connect-block Jacobi of
  // BuildPreconditioner(EBlockJacobi): blocks of one connect's nstate
  // equations (the connects of order <= 2 carry one shape)
  const bool block = prm.precond == PZG_PRECOND_BLOCK_JACOBI;
  if (!block && prm.precond != PZG_PRECOND_JACOBI) {
    set_error("pzg_solve: PCG64 takes the point or the connect-block Jacobi preconditioner");
    return PZG_EINVAL;
  }
  // high-order meshes: blocks of the real connects (several shapes each)
  const bool vblock = block && c.hp_simplex;
  if (vblock) {
    if (c.filt) {
      set_error("pzg_solve: connect-block Jacobi of a filtered high-order system not built");
      return PZG_EUNSUP;
    }
    if (c.vbj_nblk == 0) {
      set_error("pzg_solve: connect blocks of the high-order mesh not recorded");
      return PZG_ESTATE;
    }
    PZG_TRY(dev_alloc(c.d_bjinv64, sizeof(double) * std::max<int64_t>(c.vbj_ninv, 1)));
    int *fail = c.d_flag.as<int>();
    PZG_HIP(hipMemsetAsync(fail, 0, sizeof(int), c.stream));
    hipLaunchKernelGGL(k_vbj_inv64, dim3((unsigned)((c.vbj_nblk + 3) / 4)), dim3(256), 0, c.stream, c.vbj_nblk,
                       c.d_vbj_pos.as<int64_t>(), c.d_vbj_m.as<int32_t>(), c.d_vbj_off.as<int64_t>(),
                       c.d_ia.as<int64_t>(), c.d_ja.as<int64_t>(), c.d_a.as<double>(), c.d_bjinv64.as<double>(),
                       fail);
    int hf = 0;
    PZG_HIP(hipMemcpyAsync(&hf, fail, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    if (hf) {
      set_error("pzg_solve: a connect block of K is singular or not stored whole");
      return PZG_EUNSUP;
    }
  } else if (block) {
    if (c.external_csr) {
      set_error("pzg_solve: connect-block Jacobi needs the mesh's connects");
      return PZG_EUNSUP;
    }
    PZG_TRY(dev_alloc(c.d_bjinv64, sizeof(double) * c.nb * c.bs * c.bs));
    int *fail = c.d_flag.as<int>();
    PZG_HIP(hipMemsetAsync(fail, 0, sizeof(int), c.stream));
    DISPATCH_BS(c.bs, hipLaunchKernelGGL(k_bj_inv64<BS>, dim3((unsigned)((c.nb + TPB - 1) / TPB)), dim3(TPB), 0,
                                         c.stream, c.nb, c.d_ia.as<int64_t>(), c.d_a.as<double>(),
                                         c.d_bjinv64.as<double>(), fail));
    int hf = 0;
    PZG_HIP(hipMemcpyAsync(&hf, fail, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    if (hf) {
      set_error("pzg_solve: a connect block of K is singular");
      return PZG_EUNSUP;
    }
  }
  const double *dg = block ? nullptr : c.d_diag.as<double>();
  hipLaunchKernelGGL(k_cg_init64, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_f.as<double>(),
                     c.d_u.as<double>(), c.d_r.as<double>(), c.d_z.as<double>(),
                     c.d_p.as<double>(), dg, sc, part);
  hipLaunchKernelGGL(k_fin_cg_init64, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gv);
  if (vblock) {
    hipLaunchKernelGGL(k_vbj_apply64, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_vbj_eqb.as<int32_t>(),
                       c.d_vbj_pos.as<int64_t>(), c.d_vbj_m.as<int32_t>(), c.d_vbj_off.as<int64_t>(),
                       (const double *)c.d_bjinv64.as<double>(), (const double *)c.d_r.as<double>(),
                       c.d_z.as<double>(), c.d_p.as<double>(), (const SolveScalars *)nullptr, part);
    hipLaunchKernelGGL(k_bj_rho64, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gv);
  } else if (block) {
    DISPATCH_BS(c.bs, hipLaunchKernelGGL(k_bj_apply64<BS>, dim3(gv), dim3(TPB), 0, c.stream, c.nb,
                                         c.d_bjinv64.as<double>(), c.d_r.as<double>(), c.d_z.as<double>(),
                                         c.d_p.as<double>(), part));
    hipLaunchKernelGGL(k_bj_rho64, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gv);
  }
  PZG_HIP(hipGetLastError());
  int rc = PZG_OK;
  DISPATCH_BS(c.bs, rc = pcg64_iterate<BS>(c, prm, vblock ? PRE_VBLOCK : block ? PRE_BLOCK : PRE_JACOBI, hs));
  PZG_TRY(rc);
  PZG_HIP(hipEventRecord(c.ev1, c.stream));
  PZG_HIP(hipEventSynchronize(c.ev1));
  float ms = 0;
  PZG_HIP(hipEventElapsedTime(&ms, c.ev0, c.ev1));
  info.solve_ms = ms;
  info.iterations = hs.iter;
  info.outer = 1;
  info.achieved = hs.resid;
  info.converged = hs.done == 1;
  double tr = 0;
  PZG_TRY(true_residual(c, c.d_u.as<double>(), &tr));
  info.true_residual = tr;
  return hs.done == 1 ? PZG_OK : PZG_ENOCONV;
}

// ----------------------------------------------------------------------------
// Mixed path.

// q = S p; pq = p.q; pr = p.r; alpha = pr/pq
template <int BS>
__global__ __launch_bounds__(TPB) void k_fcg_spmv(int64_t nb, const int64_t *__restrict__ bia,
                                                  const int32_t *__restrict__ bja,
                                                  const float *__restrict__ v,
                                                  const float *__restrict__ p,
                                                  const float *__restrict__ r,
                                                  float *__restrict__ q, SolveScalars *sc,
                                                  double *partials) {
  if (sc->done) return;
  const int sub = threadIdx.x % BSR_L;
  int64_t lo, hi;
  int xi, xg;
  constexpr int RPB = TPB / BSR_L;  // rows per workgroup tile
#if PZG_XCD_INTERLEAVE
  xcd_slab(nb, lo, hi, xi, xg);
  const int64_t first = lo + (int64_t)xi * RPB, step = (int64_t)xg * RPB;
#else
  xcd_block_range(nb, lo, hi);
  xi = xg = 0;
  const int64_t first = lo, step = RPB;
#endif
  double pq = 0., pr = 0.;
  for (int64_t A = first + threadIdx.x / BSR_L; A < hi; A += step) {
    float out[BS];
    bsr_row<float, BS>(A, bia, bja, v, p, sub, out);
    if (sub < BS) {
      const float o = pick<float, BS>(out, sub);
      const int64_t i = A * BS + sub;
      q[i] = o;
      pq += (double)o * p[i];
      pr += (double)p[i] * r[i];
    }
  }
  double vv[2] = {pq, pr};
  block_partials<2>(vv, partials);
}

// x += alpha p; r -= alpha q; rr (slot 0); with binv z = Binv r (block Jacobi)
// and z.q (slot 1), else z is left to the preconditioner's own kernels.
// alpha = (p.r)/(p.q) from the product's partials (slots 3 and 2).
template <int BS>
__global__ __launch_bounds__(1024) void k_fcg_update(int64_t nb, float *__restrict__ x,
                                                     float *__restrict__ r, float *__restrict__ z,
                                                     const float *__restrict__ p,
                                                     const float *__restrict__ q,
                                                     const float *__restrict__ binv,
                                                     SolveScalars *A, const SolveScalars *B,
                                                     double *partials, int npq) {
  if (B->done) {
    close_step(A, B, B->pq, 0);
    return;
  }
  const int slot[2] = {2, 3}, cnt[2] = {npq, npq};
  double t[2];
  sum_slots<2>(partials, slot, cnt, t);
  const float alpha = (float)(t[1] / t[0]);
  double rr = 0., zq = 0.;
  for (int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; R < nb; R += (int64_t)gridDim.x * blockDim.x) {
    float rv[BS], qv[BS];
#pragma unroll
    for (int k = 0; k < BS; k++) {
      const int64_t i = R * BS + k;
      qv[k] = q[i];
      x[i] += alpha * p[i];
      rv[k] = r[i] - alpha * qv[k];
      r[i] = rv[k];
      rr += (double)rv[k] * rv[k];
    }
    if (!binv) continue;
    const float *bi = binv + R * BS * BS;
#pragma unroll
    for (int k = 0; k < BS; k++) {
      float u = 0.f;
#pragma unroll
      for (int l = 0; l < BS; l++) u += bi[k * BS + l] * rv[l];
      z[R * BS + k] = u;
      zq += (double)u * qv[k];
    }
  }
  if (binv) {
    double vv[2] = {rr, zq};
    store_slots<2>(vv, partials);
  } else {
    double vv[1] = {rr};
    store_slots<1>(vv, partials);
  }
  close_step(A, B, t[0], 3);
}

// Stop test on |r| before the multigrid cycle of a restarted FCG (one block;
// update due = 5: no kernel of this iteration is left to run): the restart
// recomputes z, so the last cycle of every refinement step is not run (3 of 23
// cycles on a 256^2 Darcy solve, 3 of 87 at 48^3, 3 of 38 at 64^3 with the
// learned smoother).
__global__ void k_fin_fcg_stop(SolveScalars *sc, const double *partials, int nblk) {
  if (sc->done) return;
  const double rr = sum_partials(partials, 0, nblk);
  if (threadIdx.x == 0) {
    int64_t it = sc->iter + 1;
    sc->iter = it;
    double rn = sqrt(rr);
    double resid = rn / sc->normb;
    // divergence guard: leave the loop, the host restarts from the true residual
    if (!(resid == resid) || resid > 1e3) sc->done = 3;
    else if (rn < sc->delta * sc->rlast) sc->done = 5;
    else if (it >= sc->maxit) sc->done = 2;
    sc->resid = resid;
    sc->pend = 2;
  }
}

// p = z + beta p; with pt: also pt = D^-1/2 p (input of the matrix-free
// operator).  An update request (4) still completes its direction.
__global__ __launch_bounds__(1024) void k_fcg_dir32(int64_t n, const float *__restrict__ z, float *__restrict__ p,
                                                    const float *__restrict__ dis, float *__restrict__ pt,
                                                    const SolveScalars *A, SolveScalars *B, const double *partials,
                                                    int n0, int n1) {
  double bt;
  bool upd;
  if (!next_direction<true>(A, B, partials, n0, n1, &bt, &upd) || !upd) return;
  const float beta = (float)bt;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  if (pt) {
    for (; i < n; i += st) {
      const float v = z[i] + beta * p[i];
      p[i] = v;
      pt[i] = v * dis[i];
    }
  } else {
    for (; i < n; i += st) p[i] = z[i] + beta * p[i];
  }
}

// the stored operator with the direction formed inside the product (as
// k_pcg_step64): p = z + beta p_old, q = S p, p.q and p.r (slots 2 and 3)
template <int BS>
__global__ __launch_bounds__(TPB) void k_fcg_step32(int64_t nb, const int64_t *__restrict__ bia,
                                                    const int32_t *__restrict__ bja,
                                                    const float *__restrict__ v, const float *__restrict__ z,
                                                    const float *__restrict__ p_old, float *__restrict__ p_new,
                                                    const float *__restrict__ r, float *__restrict__ q,
                                                    const SolveScalars *A, SolveScalars *B, double *partials, int n0,
                                                    int n1) {
  double bt;
  bool upd;
  if (!next_direction<true>(A, B, partials, n0, n1, &bt, &upd)) return;
  const float beta = (float)bt;
  const int sub = threadIdx.x % BSR_L;
  constexpr int RPB = TPB / BSR_L;
  double pq = 0., pr = 0.;
  auto dir = [=](int64_t i) { return upd ? z[i] + beta * p_old[i] : p_old[i]; };
  for (int64_t R = (int64_t)blockIdx.x * RPB + threadIdx.x / BSR_L; R < nb; R += (int64_t)gridDim.x * RPB) {
    float out[BS];
    bsr_row_f<float, BS>(R, bia, bja, v, dir, sub, out);
    if (sub < BS) {
      const int64_t i = R * BS + sub;
      const float o = pick<float, BS>(out, sub), pi = dir(i);
      q[i] = o;
      p_new[i] = pi;
      pq += (double)o * pi;
      pr += (double)pi * r[i];
    }
  }
  double vv[2] = {pq, pr};
  store_slots<2>(vv, partials + 2 * MAXBLK);
}

// b = D^-1/2 r64 (fp32); x = 0; r = b; z = Binv r; p = z; normb = |b|
template <int BS>
__global__ __launch_bounds__(TPB) void k_fcg_init(int64_t nb, const double *__restrict__ r64,
                                                  const double *__restrict__ dis,
                                                  float *__restrict__ x, float *__restrict__ r,
                                                  float *__restrict__ z, float *__restrict__ p,
                                                  const float *__restrict__ binv,
                                                  SolveScalars *sc, double *partials) {
  double bb = 0.;
  int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; A < nb; A += st) {
    float rv[BS];
    for (int k = 0; k < BS; k++) {
      const int64_t i = A * BS + k;
      double bi = r64[i] * dis[i];
      rv[k] = (float)bi;
      r[i] = rv[k];
      x[i] = 0.f;
      bb += bi * bi;
    }
    if (!binv) continue;  // z and p come from the multigrid cycle
    const float *bi = binv + A * BS * BS;
    for (int k = 0; k < BS; k++) {
      float s = 0.f;
      for (int l = 0; l < BS; l++) s += bi[k * BS + l] * rv[l];
      z[A * BS + k] = s;
      p[A * BS + k] = s;
    }
  }
  double vv[1] = {bb};
  block_partials<1>(vv, partials);
}
__global__ void k_fin_fcg_init(SolveScalars *sc, const double *partials, int nblk) {
  const double bb = sum_partials(partials, 0, nblk);
  if (threadIdx.x == 0) {
    double nbv = sqrt(bb);
    sc->normb = nbv > 0. ? nbv : 1.;
    sc->rlast = nbv;
    sc->resid = nbv > 0. ? 1. : 0.;
    sc->pend = 0;  // p = z follows from the start kernels
    sc->done = nbv > 0. ? 0 : 1;
  }
}

// u += D^-1/2 y; y = 0
__global__ void k_ir_update(int64_t n, float *__restrict__ y, const double *__restrict__ dis,
                            double *__restrict__ u) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    u[i] += dis[i] * (double)y[i];
    y[i] = 0.f;
  }
}

// reliable update: r = D^-1/2 r64 replaces the recursive residual; the search
// direction p is kept
__global__ __launch_bounds__(TPB) void k_fcg_reset(int64_t n, const double *__restrict__ r64,
                                                   const double *__restrict__ dis,
                                                   float *__restrict__ r, double *partials) {
  double bb = 0.;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    float v = (float)(r64[i] * dis[i]);
    r[i] = v;
    bb += (double)v * v;
  }
  double vv[1] = {bb};
  block_partials<1>(vv, partials);
}
__global__ void k_fin_fcg_reset(SolveScalars *sc, const double *partials, int nblk, double delta) {
  const double bb = sum_partials(partials, 0, nblk);
  if (threadIdx.x == 0) {
    sc->rlast = sqrt(bb);
    sc->delta = delta;
    sc->done = 0;
  }
}



int launch_spmv_bsr(Ctx &c, const float *x, float *y) {
  DISPATCH_BS(c.bs, hipLaunchKernelGGL((k_spmv_bsr<float, BS>), dim3(bsr_grid(c.nb)), dim3(TPB), 0,
                                       c.stream, c.nb, c.d_fbia.as<int64_t>(),
                                       c.d_fbja.as<int32_t>(), c.d_bsr.as<float>(), x, y));
  PZG_HIP(hipGetLastError());
  return PZG_OK;
}

constexpr int64_t FCG_MERGE_NNZ = PCG_MERGE_NNZ;
constexpr int64_t MG_INNER_CAP = 2000;  // FP32 iterations per refinement step, multigrid paths

template <int BS>
static int mixed_impl(Ctx &c, const pzg_solve_params &prm, pzg_solve_info &info) {
  const int64_t n = c.neq, nb = c.nb;
  PZG_TRY(prepare_k64(c));
  // operator of the FP32 iterations
  bool use_mf = false;
  if (prm.inner_op == PZG_INNER_MATFREE) {
    if (!mf_available(c)) {
      set_error("pzg_solve: the matrix-free inner operator needs a mesh-built system");
      return PZG_ESTATE;
    }
    use_mf = true;
  } else if (prm.inner_op == PZG_INNER_AUTO) {
    use_mf = mf_available(c);
  } else if (prm.inner_op != PZG_INNER_BSR) {
    set_error("pzg_solve: unknown inner operator");
    return PZG_EINVAL;
  }
  // the stored FP32 values of S only for the stored operator (the
  // matrix-free one needs D^-1/2 and the block-Jacobi inverses alone)
  if (use_mf) PZG_TRY(mf_prepare(c));
  else if (!c.bsr_valid) PZG_TRY(launch_build_bsr(c, true));
  PZG_TRY(ensure_reduce(c));
  // the learned preconditioner is the multigrid cycle with the learned
  // element smoother on the p level
  const bool multigrid = prm.precond == PZG_PRECOND_MULTIGRID || prm.precond == PZG_PRECOND_LEARNED;
  for (DevBuf *b : {&c.d_u, &c.d_r}) PZG_TRY(dev_alloc(*b, n * sizeof(double)));
  for (DevBuf *b : {&c.d_xs, &c.d_rs, &c.d_zs, &c.d_ps, &c.d_qs}) PZG_TRY(dev_alloc(*b, n * sizeof(float)));
  double *out = c.d_res2.as<double>();
  SolveScalars *sc = c.d_scal.as<SolveScalars>();
  double *part = c.d_partials.as<double>();
  const int gv = grid_for(n, TPB), gb = grid_for(nb, TPB), gs = bsr_grid(nb);
  const CgGrid gu = cg_grid(nb), gd = cg_grid(n);
  const int gm = std::min(gs, CG_MAXBLK);
  const int nfin = gb;  // grid of the cycle's last kernel, which forms z.q
  SolveScalars *sb = sc + 1;
  // direction formed inside the stored product (two launches an iteration);
  // the reliable update keeps the direction across batches, so it takes the
  // separate launch
  const bool merge = !use_mf && !multigrid && prm.refine == 0 && c.nbf * BS * BS <= FCG_MERGE_NNZ;
  if (merge) PZG_TRY(dev_alloc(c.d_ps2, n * sizeof(float)));
  PZG_HIP(hipEventRecord(c.ev0, c.stream));
  hipLaunchKernelGGL(k_axpby64, dim3(gv), dim3(TPB), 0, c.stream, n, 0.0, c.d_f.as<double>(), 0.0,
                     (const double *)nullptr, c.d_u.as<double>());
  int64_t total_it = 0;
  int outer = 0;
  double rel = 1.0, fnorm = 0.;
  bool conv = false;
  // a multigrid iteration costs several operator applications: short batches
  const int batch = ((prm.check_every > 0 ? prm.check_every : (multigrid ? 4 : 50)) + 1) / 2 * 2;
  auto true_res = [&](bool u_zero = false) -> int {
    if (u_zero)  // the starting guess: no product needed
      hipLaunchKernelGGL(k_residual_zero, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_f.as<double>(),
                         c.d_r.as<double>(), part);
    else
      PZG_TRY(launch_residual64(c, c.d_u.as<double>(), c.d_r.as<double>(), part, out));
    if (u_zero) fin_residual64(c, part, gv, 1, out);
    double h[2];
    PZG_HIP(hipMemcpyAsync(h, out, sizeof(h), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    rel = h[1] > 0 ? std::sqrt(h[0] / h[1]) : std::sqrt(h[0]);
    fnorm = std::sqrt(h[1]);
    return PZG_OK;
  };
  auto next_delta = [&]() {
    // reduction asked of the FP32 recursion before the next true residual
    double d = prm.inner_tol > 0 ? prm.inner_tol : 1e-4;
    double need = 0.5 * prm.tol / rel;
    if (need > d) d = need;
    return d > 0.5 ? 0.5 : d;
  };
  PZG_TRY(true_res(true));
  if (rel <= prm.tol) conv = true;
  // block Jacobi on a high-order mesh: the real connects' blocks (several
  // shapes each), inverted in FP64 and scaled into the FP32 system
  const bool vbj = prm.precond == PZG_PRECOND_BLOCK_JACOBI && c.hp_simplex && c.vbj_nblk > 0 && !c.filt;
  if (vbj && !conv) {
    PZG_TRY(dev_alloc(c.d_vbjinv64, sizeof(double) * std::max<int64_t>(c.vbj_ninv, 1)));
    PZG_TRY(dev_alloc(c.d_vbjinv32, sizeof(float) * std::max<int64_t>(c.vbj_ninv, 1)));
    int *fail = c.d_flag.as<int>();
    PZG_HIP(hipMemsetAsync(fail, 0, sizeof(int), c.stream));
    hipLaunchKernelGGL(k_vbj_inv64, dim3((unsigned)((c.vbj_nblk + 3) / 4)), dim3(256), 0, c.stream, c.vbj_nblk,
                       c.d_vbj_pos.as<int64_t>(), c.d_vbj_m.as<int32_t>(), c.d_vbj_off.as<int64_t>(),
                       c.d_ia.as<int64_t>(), c.d_ja.as<int64_t>(), c.d_a.as<double>(), c.d_vbjinv64.as<double>(),
                       fail);
    hipLaunchKernelGGL(k_vbj_scale32, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_vbj_eqb.as<int32_t>(),
                       c.d_vbj_pos.as<int64_t>(), c.d_vbj_m.as<int32_t>(), c.d_vbj_off.as<int64_t>(),
                       (const double *)c.d_vbjinv64.as<double>(), c.d_dinvsqrt.as<double>(),
                       c.d_vbjinv32.as<float>());
    int hf = 0;
    PZG_HIP(hipMemcpyAsync(&hf, fail, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    if (hf) {
      set_error("pzg_solve: a connect block of K is singular or not stored whole");
      return PZG_EUNSUP;
    }
  }
  auto vbj_apply = [&](float *z, float *p, const float *q) {
    hipLaunchKernelGGL(k_vbj_apply32, dim3(gb), dim3(TPB), 0, c.stream, n, c.d_vbj_eqb.as<int32_t>(),
                       c.d_vbj_pos.as<int64_t>(), c.d_vbj_m.as<int32_t>(), c.d_vbj_off.as<int64_t>(),
                       (const float *)c.d_vbjinv32.as<float>(), (const float *)c.d_rs.as<float>(), z, p, q,
                       (const SolveScalars *)sc, part);
  };
  if (multigrid && !conv) {
    // levels and eigenvalue estimates (timed with the solve)
    const bool les = prm.precond == PZG_PRECOND_LEARNED;
    // the learned smoother covers a wider interval (64^3 elasticity: 146 ms
    // per step at 60 against 152 ms at 30, the same at 100)
    c.mg_degree = prm.mg_degree > 0 ? prm.mg_degree : 2;
    c.mg_range = prm.mg_range > 0 ? prm.mg_range : les ? 60. : 30.;
    if (!c.mg_ready || c.mg_use_mf != use_mf || c.mg_les != les || (!c.mg_ext && mg_levels(c) < c.mg.size())) {
      c.mg_les = les;
      PZG_TRY(mg_setup(c, use_mf, true));
    }
    if (les && !c.pen_ready) PZG_TRY(pen_setup(c));
  }
  bool restart = true;
  bool learned = prm.precond == PZG_PRECOND_LEARNED;
  // PZG_TRACE=1: one line per refinement step on stderr
  const char *tr = std::getenv("PZG_TRACE");
  const bool trace = tr && tr[0] == '1';
  // learned path: the penalty rows are solved in FP64 here, after every fold,
  // to a tenth of the target residual; the FP32 iterations leave them alone
  const bool pen_rows = learned && !conv && c.pen_ready && c.pen_n > 0;
  // The penalty solve keeps d_r the exact residual f - K u (it subtracts
  // K delta on the rows that the penalized unknowns reach) and returns its
  // norm; rel_exact turns false only where an estimate stands in for it.
  int64_t pen_its = 0;
  bool rel_exact = true;
  auto pen_fix = [&]() -> int {
    pen_its = 0;
    if (!pen_rows || rel <= prm.tol) return PZG_OK;
    double p0 = 0., p1 = 0., rrf = -1.;
    // to a tenth of the target, or of what the other rows still carry
    const double tot2 = rel * rel * fnorm * fnorm;
    PZG_TRY(pen_solve(c, c.d_r.as<double>(), c.d_u.as<double>(), 0.1 * prm.tol * fnorm, prm.use_graph != 0,
                      &pen_its, &p0, &p1, 0.1, tot2, &rrf));
    if (pen_its == 0) return PZG_OK;  // u unchanged
    // without the exact update: the estimate with the -K_ip d change left out
    const double rr = rrf >= 0. ? rrf : std::max(tot2 - p0 + p1, p1);
    rel = std::sqrt(rr) / (fnorm > 0 ? fnorm : 1.);
    rel_exact = rrf >= 0.;
    return PZG_OK;
  };
  // the test on the estimate, confirmed by a true residual
  auto converged = [&](bool &cv) -> int {
    cv = false;
    if (rel > prm.tol) return PZG_OK;
    if (!rel_exact) {
      PZG_TRY(true_res());
      rel_exact = true;
    }
    cv = rel <= prm.tol;
    return PZG_OK;
  };
  PZG_TRY(pen_fix());
  PZG_TRY(converged(conv));
  int fallback = 0, stall = 0;
  double prev_rel = rel;
  SolveScalars hs;
  std::memset(&hs, 0, sizeof(hs));
  while (!conv) {
    if (restart) {
      hs.done = 0;
      hs.iter = total_it;
      // a multigrid-preconditioned inner solve takes tens of iterations: one
      // that runs past MG_INNER_CAP has stalled (the refinement step below
      // then sees no progress and falls back)
      hs.maxit = multigrid ? std::min<int64_t>(prm.max_iter, total_it + MG_INNER_CAP) : prm.max_iter;
      hs.delta = next_delta();
      PZG_HIP(hipMemcpyAsync(c.d_scal.p, &hs, sizeof(hs), hipMemcpyHostToDevice, c.stream));
      hipLaunchKernelGGL(k_fcg_init<BS>, dim3(gb), dim3(TPB), 0, c.stream, nb, c.d_r.as<double>(),
                         c.d_dinvsqrt.as<double>(), c.d_xs.as<float>(), c.d_rs.as<float>(),
                         c.d_zs.as<float>(), c.d_ps.as<float>(),
                         multigrid ? (const float *)nullptr : c.d_bjinv.as<float>(), sc, part);
      hipLaunchKernelGGL(k_fin_fcg_init, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gb);
      PZG_HIP(hipGetLastError());
      if (pen_rows) PZG_TRY(pen_zero32(c, c.d_rs.as<float>()));
      if (multigrid)
        PZG_TRY(mg_apply(c, c.d_rs.as<float>(), c.d_zs.as<float>(), c.d_ps.as<float>(), nullptr, sc, part));
      if (vbj) vbj_apply(c.d_zs.as<float>(), c.d_ps.as<float>(), nullptr);
      if (use_mf) PZG_TRY(mf_scale(c, c.d_ps.as<float>(), sc));
      restart = false;
    }
    auto step = [&](const float *p_old, float *p_new) {
      const bool early = multigrid && prm.refine == 0;
      const int n1 = multigrid ? nfin : vbj ? gb : gu.blocks;
      float *p = merge ? p_new : c.d_ps.as<float>();
      int ga = merge ? gm : gs;
      if (merge) {
        hipLaunchKernelGGL(k_fcg_step32<BS>, dim3(gm), dim3(TPB), 0, c.stream, nb, c.d_fbia.as<int64_t>(),
                           c.d_fbja.as<int32_t>(), c.d_bsr.as<float>(), (const float *)c.d_zs.as<float>(), p_old,
                           p_new, (const float *)c.d_rs.as<float>(), c.d_qs.as<float>(), (const SolveScalars *)sc, sb,
                           part, gu.blocks, n1);
      } else {
        hipLaunchKernelGGL(k_fcg_dir32, dim3(gd.blocks), dim3(gd.tpb), 0, c.stream, n,
                           (const float *)c.d_zs.as<float>(), p, use_mf ? c.d_mf_dis.as<float>() : nullptr,
                           use_mf ? c.d_mf_pt.as<float>() : nullptr, (const SolveScalars *)sc, sb,
                           (const double *)part, gu.blocks, n1);
        if (use_mf)
          (void)mf_apply(c, p, c.d_rs.as<float>(), c.d_qs.as<float>(), sb, part + 2 * MAXBLK, &ga, true);
        else
          hipLaunchKernelGGL(k_fcg_spmv<BS>, dim3(gs), dim3(TPB), 0, c.stream, nb, c.d_fbia.as<int64_t>(),
                             c.d_fbja.as<int32_t>(), c.d_bsr.as<float>(), (const float *)p, c.d_rs.as<float>(),
                             c.d_qs.as<float>(), sb, part + 2 * MAXBLK);
      }
      hipLaunchKernelGGL(k_fcg_update<BS>, dim3(gu.blocks), dim3(gu.tpb), 0, c.stream, nb, c.d_xs.as<float>(),
                         c.d_rs.as<float>(), c.d_zs.as<float>(), (const float *)p, (const float *)c.d_qs.as<float>(),
                         multigrid || vbj ? (const float *)nullptr : c.d_bjinv.as<float>(), sc,
                         (const SolveScalars *)sb, part, ga);
      // S couples the penalty rows to the others (at the 1/sqrt(big) level):
      // keep their residual at zero rather than let it drift
      if (pen_rows) (void)pen_zero32(c, c.d_rs.as<float>());
      if (early) hipLaunchKernelGGL(k_fin_fcg_stop, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gu.blocks);
      if (multigrid)
        (void)mg_apply(c, c.d_rs.as<float>(), c.d_zs.as<float>(), nullptr, c.d_qs.as<float>(), sc, part);
      if (vbj) vbj_apply(c.d_zs.as<float>(), nullptr, c.d_qs.as<float>());
    };
    auto enqueue = [&]() {
      float *p0 = c.d_ps.as<float>(), *p1 = merge ? c.d_ps2.as<float>() : p0;
      for (int k = 0; k < batch; k += 2) {
        step(p0, p1);
        step(p1, p0);
      }
      hipLaunchKernelGGL(k_cg_close<true>, dim3(1), dim3(TPB), 0, c.stream, sc, sb, (const double *)part, gu.blocks,
                         multigrid ? nfin : vbj ? gb : gu.blocks);
    };
    // the cycle's launches hold coefficients of this assembly: its graph is
    // not kept beyond the solve
    std::vector<uint64_t> key;
    if (!multigrid) {
      key_add(key, 32, BS, batch, n, nb, c.nbf, merge, use_mf, vbj);
      for (const DevBuf *b : {&c.d_scal, &c.d_partials, &c.d_xs, &c.d_rs, &c.d_zs, &c.d_ps, &c.d_ps2, &c.d_qs,
                              &c.d_bjinv, &c.d_bsr, &c.d_fbia, &c.d_fbja, &c.d_vbj_eqb, &c.d_vbj_pos, &c.d_vbj_m,
                              &c.d_vbj_off, &c.d_vbjinv32})
        key_add(key, *b);
      if (use_mf) mf_key(c, key);
    }
    PZG_TRY(run_batches(c, prm.use_graph != 0, key, enqueue, hs));
    total_it = hs.iter;
    // fold the FP32 correction into the FP64 solution and recompute the true residual
    hipLaunchKernelGGL(k_ir_update, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_xs.as<float>(),
                       c.d_dinvsqrt.as<double>(), c.d_u.as<double>());
    PZG_HIP(hipGetLastError());
    PZG_TRY(true_res());
    rel_exact = true;
    const double rel_fold = rel;
    PZG_TRY(pen_fix());
    outer++;
    if (trace)
      std::fprintf(stderr, "[pzg] refinement %d: FP32 iterations %lld (stop %d), true residual %.3e"
                   " after the fold, %.3e after the penalty rows (%lld CG iterations)\n",
                   outer, (long long)total_it, hs.done, rel_fold, rel, (long long)pen_its);
    PZG_TRY(converged(conv));
    if (conv) break;
    if (hs.done == 2 && total_it >= prm.max_iter) break;
    // Stall of the FP32 iterations (the true residual no longer halves over
    // three refinement steps, or the refinement budget is spent; with the
    // learned preconditioner already when one step gains less than 10%):
    // continue with plain FP64 Jacobi-PCG from the current solution, judged
    // by the true FP64 residual.
    stall = rel > 0.5 * prev_rel ? stall + 1 : 0;
    if (stall >= 3 || outer >= prm.max_outer ||
        (learned && rel > 0.9 * prev_rel)) {
      fallback = 1;
      if (!rel_exact) {  // the PCG restarts from d_r: make it the true residual
        PZG_TRY(true_res());
        rel_exact = true;
      }
      if (trace) std::fprintf(stderr, "[pzg] stalled: FP64 Jacobi-PCG from residual %.3e\n", rel);
      PZG_TRY(pcg64_continue(c, prm, total_it, rel));
      conv = rel <= prm.tol;
      break;
    }
    prev_rel = rel;
    if (hs.done == 3 || prm.refine == 0) { restart = true; continue; }
    hipLaunchKernelGGL(k_fcg_reset, dim3(gv), dim3(TPB), 0, c.stream, n, c.d_r.as<double>(),
                       c.d_dinvsqrt.as<double>(), c.d_rs.as<float>(), part);
    hipLaunchKernelGGL(k_fin_fcg_reset, dim3(1), dim3(TPB), 0, c.stream, sc, (const double *)part, gv, next_delta());
    PZG_HIP(hipGetLastError());
    if (pen_rows) PZG_TRY(pen_zero32(c, c.d_rs.as<float>()));
  }
  if (!rel_exact) PZG_TRY(true_res());  // the reported residual is a true one
  PZG_HIP(hipEventRecord(c.ev1, c.stream));
  PZG_HIP(hipEventSynchronize(c.ev1));
  float ms = 0;
  PZG_HIP(hipEventElapsedTime(&ms, c.ev0, c.ev1));
  info.solve_ms = ms;
  info.iterations = total_it;
  info.outer = outer;
  info.true_residual = rel;
  info.achieved = rel;
  info.converged = conv ? 1 : 0;
  info.fallback = fallback;
  return conv ? PZG_OK : PZG_ENOCONV;
}

int solve_mixed(Ctx &c, const pzg_solve_params &prm, pzg_solve_info &info) {
  if (prm.precond == PZG_PRECOND_LEARNED && !c.les_ready) {
    set_error("pzg_solve: learned preconditioner not set up in this context");
    return PZG_ESTATE;
  }
  if (c.bs == 3) return mixed_impl<3>(c, prm, info);
  if (c.bs == 1) return mixed_impl<1>(c, prm, info);
  set_error("pzg_solve: unsupported block size for the mixed solver");
  return PZG_EUNSUP;
}

}  // namespace pzg
