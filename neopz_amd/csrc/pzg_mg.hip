// pzg_mg.hip -- multigrid preconditioner of the mixed FCG path on hexahedral
// and quadrilateral meshes whose vertices form a lattice (p <= 2; a plane
// lattice has one node in z, and every kernel treats that direction as the
// identity).
//
// Levels.  Level 0 is the FCG system S = D^-1/2 K D^-1/2 (matrix-free or
// stored, as the FCG iteration uses it).  Level 1 is the trilinear subspace:
// the hierarchical shape functions of H1 (TPZShapeCube: vertex functions are
// the trilinear ones, edge/face/interior functions vanish at the vertices)
// make it the span of the vertex functions, so its prolongation is the
// injection of vertex values and its Galerkin operator P^T K P is the
// vertex-vertex part K_vv of the assembled K, read from its upper CSR.
// In level 0's scaled unknowns the transfer carries D^1/2 at the vertex
// equations.  Level 1 is stored in lattice order as a 27-point block
// stencil.  Levels 2.. halve the lattice with trilinear prolongation and the
// Galerkin product A_c = P^T A P formed on the device, while every element
// count is even and the level is too large for the dense solve; the coarsest
// level is solved with a dense inverse when it has at most MG_MAXDENSE
// unknowns.  Where an odd element count stops the halving above that, the
// solver's cycle goes on with levels that keep the last node (fine_of);
// pzg_mg_apply alone puts a Chebyshev iteration of degree MG_COARSE_DEGREE
// from zero there, a fixed SPD polynomial in M^-1 A.
//
// Smoother: Chebyshev iteration (Saad, Iterative Methods for Sparse Linear
// Systems, 2nd ed., Alg. 12.1) of degree m on M^-1 A, M = the diagonal
// nstate x nstate blocks, on the interval [lhi/range, lhi], lhi = 1.1 x the
// largest eigenvalue estimated by CG-Lanczos; m = the requested degree on
// level 0 and 1 on the lattice levels (a second step there does not lower
// the iteration count).  Each level takes m pre- and m post-smoothing steps
// with the same polynomial and the coarsest solve is exact, so the
// preconditioner is a fixed symmetric positive definite operator.  Every kernel of the cycle leaves at once when the FCG
// iteration has stopped (graph batches run past the stop).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <thread>
#include <vector>

#include "pzg_device.h"
#include "pzg_internal.h"

namespace pzg {

namespace {

constexpr int TPB = RED_TPB;
constexpr int64_t MG_DENSE = 128;      // coarsening stops at this many unknowns
constexpr int64_t MG_MAXDENSE = 1536;  // largest dense coarsest solve
constexpr int MG_COARSE_DEGREE = 8;    // Chebyshev degree of a coarsest level beyond it
constexpr double MG_COARSE_RANGE = 100.;
constexpr int MG_LANCZOS_IT = 20;      // CG-Lanczos steps per eigenvalue estimate
constexpr int MG_LATTICE_DEGREE = 1;   // Chebyshev degree on the lattice levels

int grid1(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + TPB - 1) / TPB, 1 << 20)); }
// one thread per item (kernels without a grid-stride loop)
int gridx(int64_t n) { return (int)std::max<int64_t>(1, (n + TPB - 1) / TPB); }
int gridr(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + TPB - 1) / TPB, MAXBLK)); }

__device__ inline bool stopped(const SolveScalars *sc) { return sc && sc->done; }

// y = M^-1 x at block A: entry (A, k) of the inverse blocks at m[A*sa + k*sk]
template <int BS>
__device__ inline void minv_mul(const float *__restrict__ m, int64_t sa, int64_t sk, int64_t A,
                                const float (&x)[BS], float (&y)[BS]) {
#pragma unroll
  for (int i = 0; i < BS; i++) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < BS; j++) s += m[A * sa + (i * BS + j) * sk] * x[j];
    y[i] = s;
  }
}

// ---- Chebyshev steps (vectors [nb][BS]) --------------------------------------
// Level-0 variants also write pt = D^-1/2 d (pt != null), the input of the
// matrix-free operator's next application.
// r = b; d = c0 M^-1 b; x = d
template <int BS>
__global__ void k_cheb_init(int64_t nb, const float *__restrict__ m, int64_t sa, int64_t sk,
                            const float *__restrict__ b, float *__restrict__ x, float *__restrict__ r,
                            float *__restrict__ d, float c0, const float *__restrict__ dis,
                            float *__restrict__ pt, const SolveScalars *sc) {
  if (stopped(sc)) return;
  for (int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; A < nb;
       A += (int64_t)gridDim.x * blockDim.x) {
    float bv[BS], y[BS];
#pragma unroll
    for (int k = 0; k < BS; k++) bv[k] = b[A * BS + k];
    minv_mul<BS>(m, sa, sk, A, bv, y);
#pragma unroll
    for (int k = 0; k < BS; k++) {
      r[A * BS + k] = bv[k];
      d[A * BS + k] = c0 * y[k];
      x[A * BS + k] = c0 * y[k];
      if (pt) pt[A * BS + k] = c0 * y[k] * dis[A * BS + k];
    }
  }
}

// r = b - t (t = A x); d = c0 M^-1 r; x += d
template <int BS>
__global__ void k_cheb_restart(int64_t nb, const float *__restrict__ m, int64_t sa, int64_t sk,
                               const float *__restrict__ b, const float *__restrict__ t,
                               float *__restrict__ x, float *__restrict__ r, float *__restrict__ d,
                               float c0, const float *__restrict__ dis, float *__restrict__ pt,
                               const SolveScalars *sc) {
  if (stopped(sc)) return;
  for (int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; A < nb;
       A += (int64_t)gridDim.x * blockDim.x) {
    float rv[BS], y[BS];
#pragma unroll
    for (int k = 0; k < BS; k++) {
      rv[k] = b[A * BS + k] - t[A * BS + k];
      r[A * BS + k] = rv[k];
    }
    minv_mul<BS>(m, sa, sk, A, rv, y);
#pragma unroll
    for (int k = 0; k < BS; k++) {
      d[A * BS + k] = c0 * y[k];
      x[A * BS + k] += c0 * y[k];
      if (pt) pt[A * BS + k] = c0 * y[k] * dis[A * BS + k];
    }
  }
}

// r -= t; d = c1 d + c2 M^-1 r; x += d
template <int BS>
__global__ void k_cheb_step(int64_t nb, const float *__restrict__ m, int64_t sa, int64_t sk,
                            const float *__restrict__ t, float *__restrict__ r, float *__restrict__ d,
                            float *__restrict__ x, float c1, float c2, const float *__restrict__ dis,
                            float *__restrict__ pt, const SolveScalars *sc) {
  if (stopped(sc)) return;
  for (int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; A < nb;
       A += (int64_t)gridDim.x * blockDim.x) {
    float rv[BS], y[BS];
#pragma unroll
    for (int k = 0; k < BS; k++) {
      rv[k] = r[A * BS + k] - t[A * BS + k];
      r[A * BS + k] = rv[k];
    }
    minv_mul<BS>(m, sa, sk, A, rv, y);
#pragma unroll
    for (int k = 0; k < BS; k++) {
      const float dv = c1 * d[A * BS + k] + c2 * y[k];
      d[A * BS + k] = dv;
      x[A * BS + k] += dv;
      if (pt) pt[A * BS + k] = dv * dis[A * BS + k];
    }
  }
}

// Learned smoother on level 0 (PZG_PRECOND_LEARNED): M r is an operator of
// its own (les_apply), so a Chebyshev step splits into the residual update and
// y = M r, whose gather also applies the direction / iterate update.
// mode 0: r = b;  1: r -= t;  2: r = b - t
__global__ void k_les_res(int64_t n, int mode, const float *__restrict__ b, const float *__restrict__ t,
                          float *__restrict__ r, const SolveScalars *sc) {
  if (stopped(sc)) return;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    r[i] = mode == 0 ? b[i] : mode == 1 ? r[i] - t[i] : b[i] - t[i];
}
// ---- lattice operators ---------------------------------------------------------
struct Dims {
  int n[3];
};
// (lattices hold at most INT32_MAX nodes: 32-bit divisions)
__device__ inline void node_ijk(const Dims &D, int64_t v, int &i, int &j, int &k) {
  const uint32_t u = (uint32_t)v, q = u / (uint32_t)D.n[0];
  i = (int)(u - q * (uint32_t)D.n[0]);
  k = (int)(q / (uint32_t)D.n[1]);
  j = (int)(q - (uint32_t)k * (uint32_t)D.n[1]);
}
__device__ inline int64_t node_id(const Dims &D, int i, int j, int k) {
  return i + (int64_t)D.n[0] * (j + (int64_t)D.n[1] * k);
}

// Trilinear transfer along one direction with nf fine and nc coarse nodes: nc
// == nf leaves the direction as it is (1 or 2 nodes); an odd number of
// elements (nf even) keeps the last fine node as a coarse node of its own, at
// half the distance of the others.
// fine node of coarse node I at offset dx in {-1,0,1} and its weight
__device__ inline bool fine_of(int I, int dx, int nc, int nf, int &i, float &w) {
  i = 2 * I + dx;
  w = dx ? 0.5f : 1.f;
  if (nc == nf) {
    i = I;
    return dx == 0;
  }
  if (!(nf & 1)) {
    if (I == nc - 1) {
      i = nf - 1;
      return dx == 0;
    }
    if (i == nf - 1) return false;
  }
  return i >= 0 && i < nf;
}
// first coarse node of fine node i and their number (two: weight 1/2 each)
__device__ inline int coarse_of(int i, int nc, int nf, int &n) {
  n = 1;
  if (nc == nf) return i;
  if (!(nf & 1) && i == nf - 1) return nc - 1;
  n = (i & 1) ? 2 : 1;
  return i >> 1;
}

// The steps of a lattice level (one Chebyshev step before and after the coarse
// correction).  The start d = c0 M^-1 b comes from the kernel that forms b, so a
// level is: residual b - A d, restriction (which starts the coarser level),
// then x = d + P x_c and x + c0 M^-1 (b - A x).  On planes the last two are one
// kernel (a row reads 9 neighbours, their x formed on the way); on
// three-dimensional levels the sum is its own kernel (27 neighbours of up to 8
// coarse nodes each).  Three or four launches a level instead of six, and no
// r, t vectors.

// Entries off the lattice hold zeros, so the 9 neighbours of a plane of nodes
// are read at clamped indices without a branch: their loads are in flight
// together.  With a branch per neighbour (serialised loads): residual at 49^3
// nodes and below 20.3 us on average, now 13.7; the tails below 39 us on
// planes and 47 us from 7^3 nodes x 3, now 25.5 and 31.6.

// (A x)(v, a) over the block stencil; xf(w, i, j, k, b): entry b of node w =
// (i, j, k)
template <int BS, class X>
__device__ inline float stencil_row(const Dims &D, int64_t nn, const float *__restrict__ A, int64_t v, int a, X xf) {
  int i, j, k;
  node_ijk(D, v, i, j, k);
  float acc = 0.f;
#pragma unroll 1
  for (int dz = -1; dz <= 1; dz++) {
    const int kk = k + dz;
    if (kk < 0 || kk >= D.n[2]) continue;
    float av[9][BS], xv[9][BS];
#pragma unroll
    for (int t = 0; t < 9; t++) {
      const int ii = min(max(i + t % 3 - 1, 0), D.n[0] - 1), jj = min(max(j + t / 3 - 1, 0), D.n[1] - 1);
      const int64_t w = node_id(D, ii, jj, kk);
      const float *ap = A + ((int64_t)((dz + 1) * 9 + t) * BS * BS + a * BS) * nn + v;
#pragma unroll
      for (int b = 0; b < BS; b++) {
        av[t][b] = ap[b * nn];
        xv[t][b] = xf(w, ii, jj, kk, b);
      }
    }
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int b = 0; b < BS; b++) acc += av[t][b] * xv[t][b];
  }
  return acc;
}

// P^T r at coarse node v
template <int BS, class R>
__device__ inline void restrict_node(const Dims &C, const Dims &F, int64_t v, R rf, float (&acc)[BS]) {
  int I, J, K;
  node_ijk(C, v, I, J, K);
#pragma unroll
  for (int e = 0; e < BS; e++) acc[e] = 0.f;
  int fi[3], fj[3];
  float wi[3], wj[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    if (!fine_of(I, d - 1, C.n[0], F.n[0], fi[d], wi[d])) fi[d] = min(2 * I, F.n[0] - 1), wi[d] = 0.f;
    if (!fine_of(J, d - 1, C.n[1], F.n[1], fj[d], wj[d])) fj[d] = min(2 * J, F.n[1] - 1), wj[d] = 0.f;
  }
#pragma unroll 1
  for (int dz = -1; dz <= 1; dz++) {
    int k;
    float wk;
    if (!fine_of(K, dz, C.n[2], F.n[2], k, wk)) continue;
    float rv[9][BS];
#pragma unroll
    for (int t = 0; t < 9; t++) {
      const int64_t f = node_id(F, fi[t % 3], fj[t / 3], k);
#pragma unroll
      for (int e = 0; e < BS; e++) rv[t][e] = rf(f, e);
    }
#pragma unroll
    for (int t = 0; t < 9; t++) {
      const float w = wi[t % 3] * wj[t / 3] * wk;
#pragma unroll
      for (int e = 0; e < BS; e++) acc[e] += w * rv[t][e];
    }
  }
}

// (P x_c) at fine node (i, j, k), entry e: both coarse neighbours of every
// direction, the second with weight 0 where the node lies on the first
template <class X>
__device__ inline float prolong_value(const Dims &C, const Dims &F, int i, int j, int k, int e, X xc) {
  int ni, nj, nk;
  const int i0 = coarse_of(i, C.n[0], F.n[0], ni), j0 = coarse_of(j, C.n[1], F.n[1], nj),
            k0 = coarse_of(k, C.n[2], F.n[2], nk);
  const int i1 = i0 + ni - 1, j1 = j0 + nj - 1;
  const float a0 = ni == 2 ? 0.5f : 1.f, a1 = 1.f - a0, b0 = nj == 2 ? 0.5f : 1.f, b1 = 1.f - b0;
  float acc = 0.f;
  for (int c = 0; c < nk; c++) {
    const float v00 = xc(node_id(C, i0, j0, k0 + c), e), v10 = xc(node_id(C, i1, j0, k0 + c), e),
                v01 = xc(node_id(C, i0, j1, k0 + c), e), v11 = xc(node_id(C, i1, j1, k0 + c), e);
    acc += b0 * (a0 * v00 + a1 * v10) + b1 * (a0 * v01 + a1 * v11);
  }
  return nk == 2 ? 0.5f * acc : acc;
}

// y = A x over the 27-point block stencil (set-up and the polynomial coarse
// solve); stencil entry s = (dz+1)*9 + (dy+1)*3 + (dx+1), value (s, e) of node v
// at A[(s*BS*BS + e)*nn + v].  One thread per (node, row component a on
// grid y): the small levels are latency-bound and take BS times the threads.
template <int BS>
__global__ void k_stencil(Dims D, int64_t nn, const float *__restrict__ A, const float *__restrict__ x,
                          float *__restrict__ y, const SolveScalars *sc) {
  if (stopped(sc)) return;
  const int a = blockIdx.y;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nn; v += (int64_t)gridDim.x * blockDim.x)
    y[v * BS + a] = stencil_row<BS>(D, nn, A, v, a, [x](int64_t w, int, int, int, int e) { return x[w * BS + e]; });
}

// r = b - A d, one thread per (node, component), component on grid y
template <int BS>
__global__ void k_lat_res(Dims D, int64_t nn, const float *__restrict__ A, const float *__restrict__ b,
                          const float *__restrict__ d, float *__restrict__ r, const SolveScalars *sc) {
  if (stopped(sc)) return;
  const int a = blockIdx.y;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nn; v += (int64_t)gridDim.x * blockDim.x)
    r[v * BS + a] = b[v * BS + a] - stencil_row<BS>(D, nn, A, v, a, [d](int64_t w, int, int, int, int e) { return d[w * BS + e]; });
}

// b_c = P^T r; with m: d_c = c0 M_c^-1 b_c
template <int BS>
__global__ void k_lat_restrict(Dims C, Dims F, const float *__restrict__ r, float *__restrict__ bc,
                               const float *__restrict__ m, float c0, float *__restrict__ dc,
                               const SolveScalars *sc) {
  if (stopped(sc)) return;
  const int64_t nc = (int64_t)C.n[0] * C.n[1] * C.n[2];
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nc;
       v += (int64_t)gridDim.x * blockDim.x) {
    float acc[BS], y[BS];
    restrict_node<BS>(C, F, v, [r](int64_t f, int e) { return r[f * BS + e]; }, acc);
#pragma unroll
    for (int e = 0; e < BS; e++) bc[v * BS + e] = acc[e];
    if (!m) continue;
    minv_mul<BS>(m, 1, nc, v, acc, y);
#pragma unroll
    for (int e = 0; e < BS; e++) dc[v * BS + e] = c0 * y[e];
  }
}

// x += P x_c (x holds d), one thread per (node, component)
template <int BS>
__global__ void k_lat_prolong(Dims C, Dims F, const float *__restrict__ xc, float *__restrict__ x,
                              const SolveScalars *sc) {
  if (stopped(sc)) return;
  const int64_t n = (int64_t)F.n[0] * F.n[1] * F.n[2] * BS;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t v = t / BS;
    int i, j, k;
    node_ijk(F, v, i, j, k);
    x[t] += prolong_value(C, F, i, j, k, (int)(t - v * BS), [xc](int64_t w, int e) { return xc[w * BS + e]; });
  }
}

// out = x + c0 M^-1 (b - A x); xc: x = d + P x_c formed on the way (planes), else
// x = d as given.  A workgroup takes LAT_NT nodes, wavefronts of one component
// each (coalesced stencil reads), the residual's components exchanged through
// LDS.  With vmap (the first lattice level): the correction goes straight to
// level 0, x0(vmap[v]) += D^1/2 out.
template <int BS> constexpr int lat_nt() { return BS == 1 ? 256 : 64; }
template <int BS>
__global__ __launch_bounds__(lat_nt<BS>() * BS) void k_lat_post(Dims D, int64_t nn, const float *__restrict__ A,
                                                                const float *__restrict__ m,
                                                                const float *__restrict__ b,
                                                                const float *__restrict__ d, Dims C,
                                                                const float *__restrict__ xc, float c0,
                                                                float *__restrict__ out,
                                                                const int32_t *__restrict__ vmap,
                                                                const float *__restrict__ dsq,
                                                                float *__restrict__ x0, const SolveScalars *sc) {
  if (stopped(sc)) return;
  constexpr int NT = lat_nt<BS>();
  __shared__ float sr[BS][NT];
  const int l = threadIdx.x % NT, a = threadIdx.x / NT;
  for (int64_t v0 = (int64_t)blockIdx.x * NT; v0 < nn; v0 += (int64_t)gridDim.x * NT) {
    const int64_t v = v0 + l;
    auto xf = [&](int64_t w, int i, int j, int k, int e) {
      return d[w * BS + e] + (xc ? prolong_value(C, D, i, j, k, e, [xc](int64_t q, int f) { return xc[q * BS + f]; }) : 0.f);
    };
    float res = 0.f, y = 0.f;
    if (v < nn) res = b[v * BS + a] - stencil_row<BS>(D, nn, A, v, a, xf);
    if (BS > 1) {
      __syncthreads();
      sr[a][l] = res;
      __syncthreads();
    }
    if (v >= nn) continue;
#pragma unroll
    for (int e = 0; e < BS; e++) y += m[(int64_t)(a * BS + e) * nn + v] * (BS > 1 ? sr[e][l] : res);
    int i, j, k;
    node_ijk(D, v, i, j, k);
    const float x = xf(v, i, j, k, a) + c0 * y;
    if (vmap) x0[(int64_t)vmap[v] * BS + a] += dsq[v * BS + a] * x;
    else out[v * BS + a] = x;
  }
}

// The levels from the first whose stencil is at most MG_TAIL_BYTES down to the
// dense solve, in one workgroup: every vector in LDS, the stencils and the
// inverse read through the L2, barriers in place of launches.  Bound by that
// CU's L2 reads and the barriers: 25.5 us from 65^2 nodes down (10 launches of
// about 3.5 us apart), 15.5 us from 5^3 x 3 (7 launches), 31.6 us from 7^3 x 3
// with a dense solve of 192 (6 launches).
constexpr int MG_TAIL_MAX = 12;
constexpr int64_t MG_TAIL_BYTES = 400 * 1024;
constexpr int64_t MG_TAIL_LDS = 100 * 1024;
constexpr int MG_TAIL_TPB = 1024;
struct TailArgs {
  int nl;  // levels, the last one dense
  int n[MG_TAIL_MAX][3];
  int off[MG_TAIL_MAX];  // first of the level's three vectors in LDS (floats)
  const float *A[MG_TAIL_MAX], *m[MG_TAIL_MAX];
  float c0[MG_TAIL_MAX];
  const float *cinv, *b, *d;
  float *x;
};
template <int BS>
__global__ __launch_bounds__(MG_TAIL_TPB) void k_lat_tail(TailArgs t, const SolveScalars *sc) {
  extern __shared__ float tl[];
  if (stopped(sc)) return;
  const int tid = threadIdx.x;
  auto dims = [&](int k) { return Dims{{t.n[k][0], t.n[k][1], t.n[k][2]}}; };
  auto count = [&](int k) { return t.n[k][0] * t.n[k][1] * t.n[k][2]; };
  // vectors of level k: b, d (then x), r
  const int n0 = count(0) * BS;
  for (int i = tid; i < n0; i += MG_TAIL_TPB) {
    tl[t.off[0] + i] = t.b[i];
    if (t.nl > 1) tl[t.off[0] + n0 + i] = t.d[i];
  }
  __syncthreads();
  for (int k = 0; k + 1 < t.nl; k++) {
    const Dims D = dims(k), C = dims(k + 1);
    const int nn = count(k), nc = count(k + 1);
    float *b = tl + t.off[k], *d = b + nn * BS, *r = d + nn * BS;
    float *bc = tl + t.off[k + 1], *dc = bc + nc * BS;
    for (int i = tid; i < nn * BS; i += MG_TAIL_TPB) {
      const int v = i % nn, a = i / nn;
      r[v * BS + a] = b[v * BS + a] - stencil_row<BS>(D, nn, t.A[k], v, a, [d](int64_t w, int, int, int, int e) { return d[w * BS + e]; });
    }
    __syncthreads();
    const bool start = k + 2 < t.nl;
    for (int v = tid; v < nc; v += MG_TAIL_TPB) {
      float acc[BS], y[BS];
      restrict_node<BS>(C, D, v, [r](int64_t f, int e) { return r[f * BS + e]; }, acc);
      for (int e = 0; e < BS; e++) bc[v * BS + e] = acc[e];
      if (!start) continue;
      minv_mul<BS>(t.m[k + 1], 1, nc, v, acc, y);
      for (int e = 0; e < BS; e++) dc[v * BS + e] = t.c0[k + 1] * y[e];
    }
    __syncthreads();
  }
  {  // dense solve: 16 lanes a row
    const int k = t.nl - 1, nd = count(k) * BS;
    const float *b = tl + t.off[k];
    float *x = tl + t.off[k] + nd;
    const int lane = tid & 15;
    for (int i0 = 0; i0 < nd; i0 += MG_TAIL_TPB / 16) {
      const int i = i0 + (tid >> 4);
      float s = 0.f;
      if (i < nd)
        for (int j = lane; j < nd; j += 16) s += t.cinv[(int64_t)i * nd + j] * b[j];
      s = row16_sum(s);
      if (i < nd && lane == 0) x[i] = s;
    }
    __syncthreads();
  }
  for (int k = t.nl - 2; k >= 0; k--) {
    const Dims D = dims(k), C = dims(k + 1);
    const int nn = count(k), nc = count(k + 1);
    float *b = tl + t.off[k], *d = b + nn * BS, *r = d + nn * BS;
    const float *xc = tl + t.off[k + 1] + nc * BS;
    for (int u = tid; u < nn * BS; u += MG_TAIL_TPB) {
      int i, j, l;
      node_ijk(D, u / BS, i, j, l);
      d[u] += prolong_value(C, D, i, j, l, u % BS, [xc](int64_t w, int e) { return xc[w * BS + e]; });
    }
    __syncthreads();
    for (int i = tid; i < nn * BS; i += MG_TAIL_TPB) {
      const int v = i % nn, a = i / nn;
      r[v * BS + a] = b[v * BS + a] - stencil_row<BS>(D, nn, t.A[k], v, a, [d](int64_t w, int, int, int, int e) { return d[w * BS + e]; });
    }
    __syncthreads();
    for (int i = tid; i < nn * BS; i += MG_TAIL_TPB) {
      const int v = i % nn, a = i / nn;
      float y = 0.f;
      for (int e = 0; e < BS; e++) y += t.m[k][(int64_t)(a * BS + e) * nn + v] * r[v * BS + e];
      d[v * BS + a] += t.c0[k] * y;
    }
    __syncthreads();
  }
  for (int i = tid; i < n0; i += MG_TAIL_TPB) t.x[i] = tl[t.off[0] + n0 + i];
}

// level 0 -> level 1: b1(v) = D^1/2 (r0 - t0) at the vertex block vmap[v]; with
// m: d1 = c0 M^-1 b1
template <int BS>
__global__ void k_restrict0(int64_t nn, const int32_t *__restrict__ vmap, const float *__restrict__ dsq,
                            const float *__restrict__ r0, const float *__restrict__ t0,
                            float *__restrict__ b1, const float *__restrict__ m, float c0,
                            float *__restrict__ d1, const SolveScalars *sc) {
  if (stopped(sc)) return;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nn;
       v += (int64_t)gridDim.x * blockDim.x) {
    const int64_t A = vmap[v];
    float bv[BS], y[BS];
#pragma unroll
    for (int e = 0; e < BS; e++) b1[v * BS + e] = bv[e] = dsq[v * BS + e] * (r0[A * BS + e] - t0[A * BS + e]);
    if (!m) continue;
    minv_mul<BS>(m, 1, nn, v, bv, y);
#pragma unroll
    for (int e = 0; e < BS; e++) d1[v * BS + e] = c0 * y[e];
  }
}
// x0(vmap[v]) += D^1/2 x1(v) (a hierarchy whose first lattice level is the
// coarsest or inside the tail; else k_lat_post does it)
template <int BS>
__global__ void k_prolong0(int64_t nn, const int32_t *__restrict__ vmap, const float *__restrict__ dsq,
                           const float *__restrict__ x1, float *__restrict__ x0, const SolveScalars *sc) {
  if (stopped(sc)) return;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nn;
       v += (int64_t)gridDim.x * blockDim.x) {
    const int64_t A = vmap[v];
#pragma unroll
    for (int e = 0; e < BS; e++) x0[A * BS + e] += dsq[v * BS + e] * x1[v * BS + e];
  }
}

// x = Ainv b (dense, symmetric, nd unknowns): one wavefront per row
__global__ void k_dense(int nd, const float *__restrict__ ainv, const float *__restrict__ b,
                        float *__restrict__ x, const SolveScalars *sc) {
  if (stopped(sc)) return;
  const int i = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  if (i >= nd) return;
  float s = 0.f;
  for (int j = lane; j < nd; j += 64) s += ainv[(int64_t)i * nd + j] * b[j];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) x[i] = s;
}

// z stays the preconditioned residual; p = z (restart); z.q replaces slot 1
// of the FCG update kernel's partials (same grid)
template <int BS>
__global__ __launch_bounds__(TPB) void k_mg_finish(int64_t nb, const float *__restrict__ z,
                                                   float *__restrict__ p, const float *__restrict__ q,
                                                   const SolveScalars *sc, double *partials) {
  if (stopped(sc)) return;
  double zq = 0.;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb * BS;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float v = z[i];
    if (p) p[i] = v;
    if (q) zq += (double)v * q[i];
  }
  if (!q) return;
  __shared__ double sm[TPB / 64];
  const double t = block_sum(zq, sm);
  if (threadIdx.x == 0) partials[1 * MAXBLK + blockIdx.x] = t;
}

// ---- set-up kernels --------------------------------------------------------------
// level 1 stencil from the assembled upper CSR: block (vmap[v], vmap[w]) for
// the lattice neighbour w of v in direction s, its transpose at w in the
// opposite direction.  One wavefront per vertex v scans the upper blocks of
// its block row once: vinv maps a block to its vertex (-1 for the other
// connects).  A must hold zeros (directions off the lattice or without a
// stored block).  Reads half of the rows that a scan of the full block CSR
// reads, and that format is not needed for the cycle.
template <int BS>
__global__ void k_mg_l1(Dims D, int64_t nn, const int32_t *__restrict__ vmap, const int32_t *__restrict__ vinv,
                        const int64_t *__restrict__ ia, const double *__restrict__ a,
                        const int64_t *__restrict__ ubia, const int32_t *__restrict__ ubja,
                        float *__restrict__ A) {
  constexpr int BB = BS * BS;
  const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (v >= nn) return;
  const int64_t row = vmap[v];
  if (row < 0) return;
  int i, j, k;
  node_ijk(D, v, i, j, k);
  int64_t ra[BS];
#pragma unroll
  for (int e = 0; e < BS; e++) ra[e] = ia[row * BS + e];
  if (lane < BB) {
    const int p = lane / BS, q = lane % BS, lo = p < q ? p : q, hi = p < q ? q : p;
    A[((int64_t)13 * BB + lane) * nn + v] = (float)a[ia[row * BS + lo] + (hi - lo)];
  }
  const int64_t u0 = ubia[row], nu = ubia[row + 1] - u0;
  for (int64_t q = lane; q < nu; q += 64) {
    const int32_t w = vinv[ubja[u0 + q]];
    if (w < 0) continue;
    int ii, jj, kk;
    node_ijk(D, w, ii, jj, kk);
    const int di = ii - i, dj = jj - j, dk = kk - k;
    if (di < -1 || di > 1 || dj < -1 || dj > 1 || dk < -1 || dk > 1) continue;
    const int sd = (di + 1) + 3 * (dj + 1) + 9 * (dk + 1);
#pragma unroll
    for (int e = 0; e < BS; e++)
#pragma unroll
      for (int f = 0; f < BS; f++) {
        const float x = (float)a[ra[e] + (BS - e) + q * BS + f];
        A[((int64_t)sd * BB + e * BS + f) * nn + v] = x;
        A[((int64_t)(26 - sd) * BB + f * BS + e) * nn + w] = x;
      }
  }
}
__global__ void k_mg_zero(int64_t n, float *__restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] = 0.f;
}

// Galerkin product A_c = P^T A_f P for trilinear P, one thread per coarse
// (node, stencil entry).  Along each direction the fine nodes f of N (fine_of)
// couple to the fine nodes g of the neighbour M = N + o when |g - f| <= 1; the
// pairs are enumerated per direction.
template <int BS>
__global__ void k_mg_rap(Dims C, Dims F, const float *__restrict__ Af, float *__restrict__ Ac) {
  const int64_t nc = (int64_t)C.n[0] * C.n[1] * C.n[2];
  const int64_t nf = (int64_t)F.n[0] * F.n[1] * F.n[2];
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // one thread per (coarse node, stencil entry, block entry): the coarse
  // levels are small, so the block entries spread the work over more threads
  if (x >= nc * 27 * BS * BS) return;
  const int64_t v = x % nc;
  const int s = (int)((x / nc) % 27), e = (int)(x / (nc * 27));
  int N[3];
  node_ijk(C, v, N[0], N[1], N[2]);
  const int o[3] = {s % 3 - 1, (s / 3) % 3 - 1, s / 9 - 1};
  double acc = 0.;
  bool inside = true;
  for (int d = 0; d < 3; d++) inside &= N[d] + o[d] >= 0 && N[d] + o[d] < C.n[d];
  if (inside) {
    // per direction: fine pairs (f, g) with weights and the stencil offset g - f
    int pf[3][9], pg[3][9], np[3];
    float pw[3][9];
    for (int d = 0; d < 3; d++) {
      np[d] = 0;
      const int M = N[d] + o[d];
      for (int a = -1; a <= 1; a++) {
        int f, g;
        float wf, wg;
        if (!fine_of(N[d], a, C.n[d], F.n[d], f, wf)) continue;
        for (int b = -1; b <= 1; b++) {
          if (!fine_of(M, b, C.n[d], F.n[d], g, wg) || g - f < -1 || g - f > 1) continue;
          pf[d][np[d]] = f;
          pg[d][np[d]] = g - f;
          pw[d][np[d]] = wf * wg;
          np[d]++;
        }
      }
    }
    for (int c = 0; c < np[2]; c++)
      for (int b = 0; b < np[1]; b++)
        for (int a = 0; a < np[0]; a++) {
          const int64_t f = pf[0][a] + (int64_t)F.n[0] * (pf[1][b] + (int64_t)F.n[1] * pf[2][c]);
          const int sf = (pg[2][c] + 1) * 9 + (pg[1][b] + 1) * 3 + (pg[0][a] + 1);
          const double w = (double)pw[0][a] * pw[1][b] * pw[2][c];
          acc += w * Af[((int64_t)sf * BS * BS + e) * nf + f];
        }
  }
  Ac[((int64_t)s * BS * BS + e) * nc + v] = (float)acc;
}

// inverse of the diagonal block (stencil entry 13), stored [e*nn + v]
template <int BS>
__global__ void k_mg_minv(int64_t nn, const float *__restrict__ A, float *__restrict__ minv) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nn) return;
  double a[BS * BS];
  for (int e = 0; e < BS * BS; e++) a[e] = A[((int64_t)13 * BS * BS + e) * nn + v];
  double r[BS * BS];
  if constexpr (BS == 1) {
    r[0] = a[0] != 0. ? 1. / a[0] : 0.;
  } else {
    const double c00 = a[4] * a[8] - a[5] * a[7], c01 = a[5] * a[6] - a[3] * a[8],
                 c02 = a[3] * a[7] - a[4] * a[6];
    const double det = a[0] * c00 + a[1] * c01 + a[2] * c02;
    const double id = det != 0. ? 1. / det : 0.;
    r[0] = c00 * id;
    r[1] = (a[2] * a[7] - a[1] * a[8]) * id;
    r[2] = (a[1] * a[5] - a[2] * a[4]) * id;
    r[3] = c01 * id;
    r[4] = (a[0] * a[8] - a[2] * a[6]) * id;
    r[5] = (a[2] * a[3] - a[0] * a[5]) * id;
    r[6] = c02 * id;
    r[7] = (a[1] * a[6] - a[0] * a[7]) * id;
    r[8] = (a[0] * a[4] - a[1] * a[3]) * id;
  }
  for (int e = 0; e < BS * BS; e++) minv[(int64_t)e * nn + v] = (float)r[e];
}

// dsq(v) = 1 / dinvsqrt at the vertex block vmap[v]
template <int BS>
__global__ void k_mg_dsq(int64_t nn, const int32_t *__restrict__ vmap, const double *__restrict__ dis,
                         float *__restrict__ dsq) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nn) return;
  for (int e = 0; e < BS; e++) dsq[v * BS + e] = (float)(1.0 / dis[(int64_t)vmap[v] * BS + e]);
}

__global__ void k_hash_fill(int64_t n, float *__restrict__ v, uint64_t seed) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t h = (uint64_t)i * 0x9E3779B97F4A7C15ULL + seed;
    h ^= h >> 31;
    h *= 0xBF58476D1CE4E5B9ULL;
    h ^= h >> 29;
    v[i] = (float)((double)(h >> 11) / 9007199254740992.0) - 0.5f;
  }
}

// Chebyshev coefficients of one level
struct Cheb {
  float c0;
  std::vector<float> c1, c2;  // steps 1 .. m-1
};
Cheb cheb_coeffs(double lmax, double range, int m) {
  const double hi = 1.1 * lmax, lo = hi / range;
  const double theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo), sigma = theta / delta;
  Cheb ch;
  ch.c0 = (float)(1.0 / theta);
  double rho = 1.0 / sigma;
  for (int j = 1; j < m; j++) {
    const double rn = 1.0 / (2.0 * sigma - rho);
    ch.c1.push_back((float)(rn * rho));
    ch.c2.push_back((float)(2.0 * rn / delta));
    rho = rn;
  }
  return ch;
}

// A level for the smoother: operator, inverse diagonal blocks, vectors
struct LevelView {
  int64_t nb;              // blocks
  const float *m;          // inverse diagonal blocks
  int64_t sa, sk;          // their layout
  float *r, *d, *t;        // work vectors
  const float *dis = nullptr;  // level 0, matrix-free: D^-1/2 and the operator's
  float *pt = nullptr;         // pre-scaled input, written with each new d
  float *pt2 = nullptr;        // level 0, tiled operator: the second such buffer
  bool les = false;            // level 0: M is the learned smoother (else the blocks m)
  Cheb ch;
};

// op(x, y, prescaled): y = A x; prescaled: L.pt already holds D^-1/2 x.
// Leaves x and, as r - t, the residual b - A x (the restriction subtracts).
// the learned smoother's steps (LevelView::les)
template <int BS, class Op>
int smooth_les(Ctx &c, const LevelView &L, const float *b, float *x, Op op, const SolveScalars *sc,
               bool pre) {
  const int64_t n = L.nb * BS;
  const int g = grid1(n);
  const bool ps = L.pt != nullptr;
  if (L.pt2) {
    // the residual update in the operator's own pass (at 64^3 elements 15 us a
    // step for k_les_res and t)
    MfOut o;
    o.mode = MF_OUT_RES;
    o.dis = L.dis;
    o.rin = b;
    o.rout = L.r;
    if (!pre) {
      PZG_TRY(mf_scale(c, x, sc));
      PZG_TRY(mf_apply_out(c, o, sc));
      o.rin = L.r;
    } else if (L.ch.c1.empty()) {  // the restriction reads r
      hipLaunchKernelGGL(k_les_res, dim3(g), dim3(TPB), 0, c.stream, n, 0, b, (const float *)nullptr, L.r, sc);
    }
    LesCheb ch{pre ? 0 : 1, 0.f, (float)L.ch.c0, L.d, x, L.pt, L.dis};
    PZG_TRY(les_apply(c, o.rin, nullptr, sc, &ch));
    for (size_t j = 0; j < L.ch.c1.size(); j++) {
      PZG_TRY(mf_apply_out(c, o, sc));
      o.rin = L.r;
      LesCheb chj{2, (float)L.ch.c1[j], (float)L.ch.c2[j], L.d, x, L.pt, L.dis};
      PZG_TRY(les_apply(c, L.r, nullptr, sc, &chj));
    }
    return pre ? op(L.d, L.t, ps) : PZG_OK;
  }
  if (pre) {
    hipLaunchKernelGGL(k_les_res, dim3(g), dim3(TPB), 0, c.stream, n, 0, b, (const float *)nullptr, L.r, sc);
  } else {
    PZG_TRY(op(x, L.t, false));
    hipLaunchKernelGGL(k_les_res, dim3(g), dim3(TPB), 0, c.stream, n, 2, b, L.t, L.r, sc);
  }
  LesCheb ch{pre ? 0 : 1, 0.f, (float)L.ch.c0, L.d, x, L.pt, L.dis};
  PZG_TRY(les_apply(c, L.r, nullptr, sc, &ch));
  for (size_t j = 0; j < L.ch.c1.size(); j++) {
    PZG_TRY(op(L.d, L.t, ps));
    hipLaunchKernelGGL(k_les_res, dim3(g), dim3(TPB), 0, c.stream, n, 1, b, L.t, L.r, sc);
    LesCheb chj{2, (float)L.ch.c1[j], (float)L.ch.c2[j], L.d, x, L.pt, L.dis};
    PZG_TRY(les_apply(c, L.r, nullptr, sc, &chj));
  }
  return pre ? op(L.d, L.t, ps) : PZG_OK;
}

// The Chebyshev steps in the tiled operator's own passes: with restart (x += c0 M
// (b - S x) first) or after k_cheb_init; keep: d and pt are needed afterwards, and
// *pin then is the buffer that holds D^-1/2 d.
int steps_tiled(Ctx &c, const LevelView &L, const float *b, float *x, const SolveScalars *sc, bool restart,
                const float **pin) {
  MfOut o;
  o.mode = MF_OUT_CHEB;
  o.dis = L.dis;
  o.minv = L.m;
  o.d = L.d;
  o.x = x;
  o.rout = L.r;
  float *from = L.pt, *to = L.pt2;
  const size_t m = L.ch.c1.size();
  for (size_t j = restart ? 0 : 1; j <= m; j++) {
    const bool last = j == m && !pin;  // nothing after it reads r, d or pt
    o.rin = j == 0 ? b : L.r;
    o.rout = last ? nullptr : L.r;
    o.c1 = j == 0 ? 0.f : (float)L.ch.c1[j - 1];
    o.c2 = j == 0 ? L.ch.c0 : (float)L.ch.c2[j - 1];
    o.pin = from;
    o.pt = last ? nullptr : to;
    PZG_TRY(mf_apply_out(c, o, sc));
    std::swap(from, to);
  }
  if (pin) *pin = from;
  return PZG_OK;
}

template <int BS, class Op>
int smooth_pre(Ctx &c, const LevelView &L, const float *b, float *x, Op op, const SolveScalars *sc) {
  if (L.les) return smooth_les<BS>(c, L, b, x, op, sc, true);
  const int g = grid1(L.nb);
  const bool ps = L.pt != nullptr;
  hipLaunchKernelGGL(k_cheb_init<BS>, dim3(g), dim3(TPB), 0, c.stream, L.nb, L.m, L.sa, L.sk, b, x, L.r,
                     L.d, L.ch.c0, L.dis, L.pt, sc);
  PZG_HIP(hipGetLastError());
  if (L.pt2) {
    MfOut o;
    o.dis = L.dis;
    o.t = L.t;
    PZG_TRY(steps_tiled(c, L, b, x, sc, false, &o.pin));
    return mf_apply_out(c, o, sc);
  }
  for (size_t j = 0; j < L.ch.c1.size(); j++) {
    PZG_TRY(op(L.d, L.t, ps));
    hipLaunchKernelGGL(k_cheb_step<BS>, dim3(g), dim3(TPB), 0, c.stream, L.nb, L.m, L.sa, L.sk, L.t, L.r,
                       L.d, x, L.ch.c1[j], L.ch.c2[j], L.dis, L.pt, sc);
    PZG_HIP(hipGetLastError());
  }
  return op(L.d, L.t, ps);
}

template <int BS, class Op>
int smooth_post(Ctx &c, const LevelView &L, const float *b, float *x, Op op, const SolveScalars *sc) {
  if (L.les) return smooth_les<BS>(c, L, b, x, op, sc, false);
  const int g = grid1(L.nb);
  const bool ps = L.pt != nullptr;
  if (L.pt2) {
    PZG_TRY(mf_scale(c, x, sc));
    return steps_tiled(c, L, b, x, sc, true, nullptr);
  }
  PZG_TRY(op(x, L.t, false));
  hipLaunchKernelGGL(k_cheb_restart<BS>, dim3(g), dim3(TPB), 0, c.stream, L.nb, L.m, L.sa, L.sk, b, L.t, x,
                     L.r, L.d, L.ch.c0, L.dis, L.pt, sc);
  PZG_HIP(hipGetLastError());
  for (size_t j = 0; j < L.ch.c1.size(); j++) {
    PZG_TRY(op(L.d, L.t, ps));
    hipLaunchKernelGGL(k_cheb_step<BS>, dim3(g), dim3(TPB), 0, c.stream, L.nb, L.m, L.sa, L.sk, L.t, L.r,
                       L.d, x, L.ch.c1[j], L.ch.c2[j], L.dis, L.pt, sc);
    PZG_HIP(hipGetLastError());
  }
  return PZG_OK;
}

Dims dims_of(const MgLevel &l) { return Dims{{l.n[0], l.n[1], l.n[2]}}; }

// level-0 operator y = S x (matrix-free or stored FP32); prescaled: the
// matrix-free input D^-1/2 x is already in place
int op0(Ctx &c, const float *x, float *y, const SolveScalars *sc, bool prescaled) {
  if (c.mg_use_mf) return mf_apply(c, x, nullptr, y, sc, nullptr, nullptr, prescaled);
  return launch_spmv_bsr(c, x, y);
}

template <int BS>
int op_lattice(Ctx &c, const MgLevel &l, const float *x, float *y, const SolveScalars *sc) {
  hipLaunchKernelGGL(k_stencil<BS>, dim3(grid1(l.nn), BS), dim3(TPB), 0, c.stream, dims_of(l), l.nn,
                     l.A.as<float>(), x, y, sc);
  PZG_HIP(hipGetLastError());
  return PZG_OK;
}

LevelView view0(Ctx &c) {
  LevelView v;
  v.nb = c.nb;
  v.m = c.d_bjinv.as<float>();
  v.sa = (int64_t)c.bs * c.bs;
  v.sk = 1;
  v.r = c.d_mg_r0.as<float>();
  v.d = c.d_mg_d0.as<float>();
  v.t = c.d_mg_t0.as<float>();
  if (c.mg_use_mf) {
    v.dis = c.d_mf_dis.as<float>();
    v.pt = c.d_mf_pt.as<float>();
    if (c.mf_tile) v.pt2 = c.d_mt_pt2.as<float>();
  }
  v.les = c.mg_les;
  v.ch = cheb_coeffs(c.mg_lmax0, c.mg_range, c.mg_degree);
  return v;
}
LevelView view_l(Ctx &c, MgLevel &l) {
  LevelView v;
  v.nb = l.nn;
  v.m = l.minv.as<float>();
  v.sa = 1;
  v.sk = l.nn;
  v.r = l.r.as<float>();
  v.d = l.d.as<float>();
  v.t = l.t.as<float>();
  v.ch = cheb_coeffs(l.lmax, c.mg_range, MG_LATTICE_DEGREE);
  return v;
}

// largest eigenvalue of the symmetric tridiagonal (a, b): bisection on the
// Sturm count (eigenvalues below x = negative pivots of T - x I)
double tridiag_max(const std::vector<double> &a, const std::vector<double> &b) {
  const int k = (int)a.size();
  double hi = 0.;
  for (int i = 0; i < k; i++)
    hi = std::max(hi, a[i] + (i > 0 ? std::fabs(b[i - 1]) : 0.) + (i + 1 < k ? std::fabs(b[i]) : 0.));
  double lo = 0.;
  auto below = [&](double x) {
    int cnt = 0;
    double d = 1.;
    for (int i = 0; i < k; i++) {
      d = a[i] - x - (i > 0 ? b[i - 1] * b[i - 1] / d : 0.);
      if (d == 0.) d = -1e-300;
      if (d < 0.) cnt++;
    }
    return cnt;
  };
  for (int it = 0; it < 100; it++) {
    const double mid = 0.5 * (lo + hi);
    if (below(mid) == k) hi = mid;
    else lo = mid;
  }
  return hi;
}

// CG-Lanczos on the device.  lz[0] = r.z of the current step, lz[1 + 2k] =
// alpha_k, lz[2 + 2k] = beta_k, lz[LZ_ZERO] = 0; a step whose p.q or r.z is
// not positive leaves alpha = 0 (and every later step with it).
constexpr int LZ_ZERO = 2 * MG_LANCZOS_IT + 1;

// r -= alpha q; z = M^-1 r; partial sums of r.z (alpha = *al)
template <int BS>
__global__ __launch_bounds__(TPB) void k_lz_update(int64_t nb, const float *__restrict__ m, int64_t sa,
                                                   int64_t sk, const double *__restrict__ al,
                                                   const float *__restrict__ q, float *__restrict__ r,
                                                   float *__restrict__ z, double *partials) {
  const float alpha = (float)*al;
  double rz = 0.;
  for (int64_t A = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; A < nb;
       A += (int64_t)gridDim.x * blockDim.x) {
    float rv[BS], y[BS];
    for (int k = 0; k < BS; k++) {
      rv[k] = r[A * BS + k] - alpha * q[A * BS + k];
      r[A * BS + k] = rv[k];
    }
    minv_mul<BS>(m, sa, sk, A, rv, y);
    for (int k = 0; k < BS; k++) {
      z[A * BS + k] = y[k];
      rz += (double)rv[k] * y[k];
    }
  }
  double vv[1] = {rz};
  block_partials<1>(vv, partials);
}
__global__ __launch_bounds__(TPB) void k_dot(int64_t n, const float *__restrict__ a,
                                             const float *__restrict__ b, double *partials) {
  double s = 0.;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    s += (double)a[i] * b[i];
  double vv[1] = {s};
  block_partials<1>(vv, partials);
}
// one block: what = 0: lz[0] = r.z; 1: alpha_k = lz[0] / p.q; 2: beta_k =
// r.z / lz[0], lz[0] = r.z
__global__ void k_lz_scalar(const double *partials, int nblk, double *lz, int k, int what) {
  const double s = sum_partials(partials, 0, nblk);
  if (threadIdx.x != 0) return;
  if (what == 0) {
    lz[0] = s;
  } else if (what == 1) {
    const bool live = k == 0 || lz[1 + 2 * (k - 1)] > 0.;
    lz[1 + 2 * k] = live && s > 0. && lz[0] > 0. ? lz[0] / s : 0.;
  } else {
    const bool live = lz[1 + 2 * k] > 0. && s > 0.;
    lz[2 + 2 * k] = live ? s / lz[0] : 0.;
    if (live) lz[0] = s;
  }
}
// p = z + beta p (beta = *be)
__global__ void k_xpby(int64_t n, const float *__restrict__ z, const double *__restrict__ be,
                       float *__restrict__ p) {
  const float beta = (float)*be;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = z[i] + beta * p[i];
}

// largest eigenvalue of M^-1 A: MG_LANCZOS_IT steps of preconditioned CG
// from a pseudo-random right-hand side, all on the device; the CG
// coefficients give the Lanczos tridiagonal (diagonal 1/alpha_k +
// beta_{k-1}/alpha_{k-1}, off-diagonal sqrt(beta_k)/alpha_k), whose largest
// eigenvalue approximates lmax from below.  Work vectors: r, z, p, q.
// r -= alpha q (alpha = *al)
__global__ void k_lz_rsub(int64_t n, const double *__restrict__ al, const float *__restrict__ q,
                          float *__restrict__ r) {
  const float alpha = (float)*al;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    r[i] -= alpha * q[i];
}

template <int BS, class Op>
int lanczos_lmax(Ctx &c, int64_t nb, const float *m, int64_t sa, int64_t sk, float *r, float *z, float *p,
                 float *q, Op op, double &lmax, bool les = false) {
  const int64_t n = nb * BS;
  double *part = c.d_partials.as<double>();
  double *lz = c.d_mg_lz.as<double>();
  const int gr = gridr(n), gb = gridr(nb);
  // r -= alpha q; z = M r; partials of r.z; returns the number of partial blocks
  auto mstep = [&](const double *al, const float *qq) -> int {
    if (!les) {
      hipLaunchKernelGGL(k_lz_update<BS>, dim3(gb), dim3(TPB), 0, c.stream, nb, m, sa, sk, al, qq, r, z, part);
      return gb;
    }
    hipLaunchKernelGGL(k_lz_rsub, dim3(grid1(n)), dim3(TPB), 0, c.stream, n, al, qq, r);
    if (les_apply(c, r, z, nullptr) != PZG_OK) return -1;
    hipLaunchKernelGGL(k_dot, dim3(gr), dim3(TPB), 0, c.stream, n, r, z, part);
    return gr;
  };
  PZG_HIP(hipMemsetAsync(lz, 0, sizeof(double) * (LZ_ZERO + 1), c.stream));
  hipLaunchKernelGGL(k_hash_fill, dim3(grid1(n)), dim3(TPB), 0, c.stream, n, r, (uint64_t)0x5DEECE66DULL);
  // z = M^-1 r and r.z (the update with alpha = 0)
  int nblk = mstep(lz + LZ_ZERO, r);
  if (nblk < 0) return PZG_EHIP;
  hipLaunchKernelGGL(k_lz_scalar, dim3(1), dim3(TPB), 0, c.stream, (const double *)part, nblk, lz, 0, 0);
  PZG_HIP(hipGetLastError());
  PZG_HIP(hipMemcpyAsync(p, z, sizeof(float) * n, hipMemcpyDeviceToDevice, c.stream));
  for (int k = 0; k < MG_LANCZOS_IT; k++) {
    PZG_TRY(op(p, q));
    hipLaunchKernelGGL(k_dot, dim3(gr), dim3(TPB), 0, c.stream, n, p, q, part);
    hipLaunchKernelGGL(k_lz_scalar, dim3(1), dim3(TPB), 0, c.stream, (const double *)part, gr, lz, k, 1);
    nblk = mstep(lz + 1 + 2 * k, q);
    if (nblk < 0) return PZG_EHIP;
    hipLaunchKernelGGL(k_lz_scalar, dim3(1), dim3(TPB), 0, c.stream, (const double *)part, nblk, lz, k, 2);
    hipLaunchKernelGGL(k_xpby, dim3(grid1(n)), dim3(TPB), 0, c.stream, n, z, lz + 2 + 2 * k, p);
    PZG_HIP(hipGetLastError());
  }
  std::vector<double> h(LZ_ZERO + 1);
  PZG_HIP(hipMemcpyAsync(h.data(), lz, sizeof(double) * h.size(), hipMemcpyDeviceToHost, c.stream));
  PZG_HIP(hipStreamSynchronize(c.stream));
  std::vector<double> ta, tb;
  for (int k = 0; k < MG_LANCZOS_IT; k++) {
    const double alpha = h[1 + 2 * k], beta = h[2 + 2 * k];
    if (!(alpha > 0.)) break;
    ta.push_back(1.0 / alpha + (k > 0 ? h[2 * k] / h[2 * k - 1] : 0.));
    if (!(beta > 0.)) break;
    tb.push_back(std::sqrt(beta) / alpha);
  }
  if (ta.empty()) {
    set_error("multigrid: operator not positive definite on a level");
    return PZG_EUNSUP;
  }
  tb.resize(ta.size());
  lmax = tridiag_max(ta, tb);
  return PZG_OK;
}

// In-place inverse of a symmetric positive definite matrix (FP64, n x n) by
// Gauss-Jordan sweeps without pivoting, one pivot per launch pair: k_gj_save
// keeps row and column k, k_gj_step applies the sweep
//   a_kk = 1/p, a_kj = a_kj/p, a_ik = -a_ik/p, a_ij -= a_ik a_kj / p
// (p = a_kk; after every pivot the array holds A^-1).  A pivot <= 0 sets
// *fail (A not positive definite).
__global__ void k_gj_save(int n, const double *__restrict__ m, int k, double *__restrict__ prow,
                          double *__restrict__ pcol) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) {
    prow[t] = m[(size_t)k * n + t];
    pcol[t] = m[(size_t)t * n + k];
  }
}
__global__ void k_gj_step(int n, double *__restrict__ m, int k, const double *__restrict__ prow,
                          const double *__restrict__ pcol, int *fail) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)n * n) return;
  const int i = (int)(t / n), j = (int)(t % n);
  const double p = prow[k];
  if (t == 0 && !(p > 0.)) *fail = 1;
  const double ip = 1. / p;
  double v;
  if (i == k) v = j == k ? ip : prow[j] * ip;
  else if (j == k) v = -pcol[i] * ip;
  else v = m[t] - pcol[i] * prow[j] * ip;
  m[t] = v;
}
__global__ void k_d2f_n(int64_t n, const double *__restrict__ a, float *__restrict__ b) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) b[t] = (float)a[t];
}

// Mesh-level part: the vertex lattice, the levels and their buffers (kept
// until the mesh changes).
template <int BS>
int structure_impl(Ctx &c) {
  mg_free(c);
  // vertex lattice: the corner nodes of the volume elements and their blocks
  const bool hex = c.dim == 3 && c.vol_etype == PZG_HEX, quad = c.dim == 2 && c.vol_etype == PZG_QUAD;
  if (!c.has_mesh || !(hex || quad) || c.hp_simplex || c.has_dep || c.external_csr) {
    set_error("multigrid preconditioner: needs a hexahedral or quadrilateral mesh-built system without "
              "constrained connects");
    return PZG_EUNSUP;
  }
  const int nc = c.vol_ncorner, nsd = c.vol_nsides;
  std::vector<int64_t> nblk(c.nnodes, -1);
  int64_t nvert = 0;
  for (int64_t e = 0; e < c.nvol; e++)
    for (int k = 0; k < nc; k++) {  // sides 0 .. nc-1: the corners
      const int64_t node = c.vol_nodes[e * nc + k];
      const int64_t b = c.aidx[c.vol_conn[e * nsd + k]];
      if (b < 0 || c.blk_size[c.vol_conn[e * nsd + k]] != BS) {
        set_error("multigrid preconditioner: a vertex connect without its own equations");
        return PZG_EUNSUP;
      }
      if (nblk[node] == -1) {
        nblk[node] = b;
        nvert++;
      } else if (nblk[node] != b) {
        set_error("multigrid preconditioner: a mesh node with two vertex connects");
        return PZG_EUNSUP;
      }
    }
  // distinct coordinates per direction (to 1e-9 of the extent)
  int n[3];
  std::vector<std::vector<double>> u(3);
  for (int d = 0; d < 3; d++) {
    std::vector<double> x;
    for (int64_t p = 0; p < c.nnodes; p++)
      if (nblk[p] >= 0) x.push_back(c.xyz[3 * p + d]);
    std::sort(x.begin(), x.end());
    const double tol = 1e-9 * std::max(1.0, std::fabs(x.back() - x.front()));
    for (double v : x)
      if (u[d].empty() || v - u[d].back() > tol) u[d].push_back(v);
    n[d] = (int)u[d].size();
  }
  const int64_t nn1 = (int64_t)n[0] * n[1] * n[2];
  if (nn1 != nvert || nn1 > INT32_MAX) {
    set_error("multigrid preconditioner: the mesh vertices do not form a lattice");
    return PZG_EUNSUP;
  }
  std::vector<int32_t> vmap(nn1, -1);
  for (int64_t p = 0; p < c.nnodes; p++) {
    if (nblk[p] < 0) continue;
    int id[3];
    for (int d = 0; d < 3; d++) {
      const double v = c.xyz[3 * p + d];
      auto it = std::lower_bound(u[d].begin(), u[d].end(), v - 1e-9 * std::max(1.0, std::fabs(u[d].back() - u[d].front())));
      id[d] = (int)(it - u[d].begin());
      if (id[d] >= n[d]) id[d] = n[d] - 1;
    }
    const int64_t l = id[0] + (int64_t)n[0] * (id[1] + (int64_t)n[1] * id[2]);
    if (vmap[l] != -1) {
      set_error("multigrid preconditioner: the mesh vertices do not form a lattice");
      return PZG_EUNSUP;
    }
    vmap[l] = (int32_t)nblk[p];
  }
  // levels: halve while the element counts are even and the level is too
  // large for the dense solve
  {
    MgLevel l;
    for (int d = 0; d < 3; d++) l.n[d] = n[d];
    l.nn = nn1;
    c.mg.push_back(std::move(l));
  }
  for (;;) {
    const MgLevel &f = c.mg.back();
    if (f.nn * BS <= MG_DENSE) break;
    // a direction of one node (the z of a plane lattice) stays as it is
    bool even = true;
    for (int d = 0; d < 3; d++) even &= f.n[d] == 1 || ((f.n[d] - 1) % 2 == 0 && f.n[d] >= 3);
    if (!even) break;
    MgLevel l;
    for (int d = 0; d < 3; d++) l.n[d] = f.n[d] == 1 ? 1 : (f.n[d] - 1) / 2 + 1;
    l.nn = (int64_t)l.n[0] * l.n[1] * l.n[2];
    c.mg.push_back(std::move(l));
  }
  c.mg_dense = c.mg.back().nn * BS <= MG_MAXDENSE;
  c.mg_nstd = c.mg.size();
  // the solver's cycle goes on where an odd count stopped the halving above
  // the dense limit: every direction with more than one element is coarsened,
  // an odd count keeping its last node (fine_of).  A 255^2 lattice (256^2
  // nodes) with the polynomial in place of these levels took 205 FCG
  // iterations, with them as many as its even neighbour.
  while (!c.mg_dense && c.mg.back().nn * BS > MG_DENSE) {
    const MgLevel &f = c.mg.back();
    MgLevel l;
    bool less = false;
    for (int d = 0; d < 3; d++) {
      l.n[d] = f.n[d] <= 2 ? f.n[d] : f.n[d] / 2 + 1;  // (odd n: (n - 1)/2 + 1)
      less |= l.n[d] < f.n[d];
    }
    if (!less) break;
    l.nn = (int64_t)l.n[0] * l.n[1] * l.n[2];
    c.mg.push_back(std::move(l));
  }
  // device arrays
  PZG_TRY(dev_upload(c.d_mg_vmap, vmap.data(), vmap.size(), c.stream));
  {
    std::vector<int32_t> vinv(c.nb, -1);  // block -> vertex of the level-1 lattice
    for (size_t w = 0; w < vmap.size(); w++)
      if (vmap[w] >= 0) vinv[vmap[w]] = (int32_t)w;
    PZG_TRY(dev_upload(c.d_mg_vinv, vinv.data(), vinv.size(), c.stream));
  }
  PZG_TRY(dev_alloc(c.d_mg_dsq, sizeof(float) * nn1 * BS));
  PZG_TRY(dev_alloc(c.d_mg_lz, sizeof(double) * (LZ_ZERO + 1)));
  for (DevBuf *b : {&c.d_mg_r0, &c.d_mg_d0, &c.d_mg_t0, &c.d_mg_w0}) PZG_TRY(dev_alloc(*b, sizeof(float) * c.neq));
  for (MgLevel &l : c.mg) {
    PZG_TRY(dev_alloc(l.A, sizeof(float) * 27 * BS * BS * l.nn));
    PZG_TRY(dev_alloc(l.minv, sizeof(float) * BS * BS * l.nn));
    for (DevBuf *b : {&l.x, &l.b, &l.r, &l.d, &l.t}) PZG_TRY(dev_alloc(*b, sizeof(float) * BS * l.nn));
  }
  PZG_HIP(hipFuncSetAttribute((const void *)k_lat_tail<BS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)MG_TAIL_LDS));
  c.mg_struct = true;
  return PZG_OK;
}

// Matrix-level part (after every assembly): D^1/2 at the vertices, the
// level operators, the coarsest inverse and the eigenvalue estimates.
template <int BS>
int setup_impl(Ctx &c) {
  if (!c.mg_struct) PZG_TRY(structure_impl<BS>(c));
  const int64_t nn1 = c.mg[0].nn;
  hipLaunchKernelGGL(k_mg_dsq<BS>, dim3(gridx(nn1)), dim3(TPB), 0, c.stream, nn1, c.d_mg_vmap.as<int32_t>(),
                     c.d_dinvsqrt.as<double>(), c.d_mg_dsq.as<float>());
  hipLaunchKernelGGL(k_mg_zero, dim3(gridr(27 * BS * BS * nn1)), dim3(TPB), 0, c.stream, 27 * BS * BS * nn1,
                     c.mg[0].A.as<float>());
  hipLaunchKernelGGL(k_mg_l1<BS>, dim3(gridx(64 * nn1)), dim3(TPB), 0, c.stream, dims_of(c.mg[0]), nn1,
                     c.d_mg_vmap.as<int32_t>(), c.d_mg_vinv.as<int32_t>(), c.d_ia.as<int64_t>(),
                     c.d_a.as<double>(), c.d_ubia.as<int64_t>(), c.d_ubja.as<int32_t>(), c.mg[0].A.as<float>());
  PZG_HIP(hipGetLastError());
  const size_t nl = mg_levels(c);
  const bool dense = mg_dense_coarse(c);
  for (size_t k = 1; k < nl; k++) {
    hipLaunchKernelGGL(k_mg_rap<BS>, dim3(gridx(27 * BS * BS * c.mg[k].nn)), dim3(TPB), 0, c.stream, dims_of(c.mg[k]),
                       dims_of(c.mg[k - 1]), c.mg[k - 1].A.as<float>(), c.mg[k].A.as<float>());
    PZG_HIP(hipGetLastError());
  }
  for (size_t k = 0; k < nl; k++) {
    MgLevel &l = c.mg[k];
    hipLaunchKernelGGL(k_mg_minv<BS>, dim3(gridx(l.nn)), dim3(TPB), 0, c.stream, l.nn, l.A.as<float>(),
                       l.minv.as<float>());
    PZG_HIP(hipGetLastError());
  }
  // dense inverse of the coarsest level
  if (dense) {
    const MgLevel &l = c.mg[nl - 1];
    const int nd = (int)(l.nn * BS);
    std::vector<float> h((size_t)27 * BS * BS * l.nn);
    PZG_HIP(hipMemcpyAsync(h.data(), l.A.p, h.size() * sizeof(float), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    std::vector<double> a((size_t)nd * nd, 0.);
    for (int64_t v = 0; v < l.nn; v++) {
      const int i = (int)(v % l.n[0]), j = (int)((v / l.n[0]) % l.n[1]), k = (int)(v / ((int64_t)l.n[0] * l.n[1]));
      for (int s = 0; s < 27; s++) {
        const int ii = i + s % 3 - 1, jj = j + (s / 3) % 3 - 1, kk = k + s / 9 - 1;
        if (ii < 0 || jj < 0 || kk < 0 || ii >= l.n[0] || jj >= l.n[1] || kk >= l.n[2]) continue;
        const int64_t w = ii + (int64_t)l.n[0] * (jj + (int64_t)l.n[1] * kk);
        for (int e = 0; e < BS * BS; e++)
          a[(size_t)(v * BS + e / BS) * nd + w * BS + e % BS] = h[((size_t)s * BS * BS + e) * l.nn + v];
      }
    }
    for (int i = 0; i < nd; i++)  // symmetric part (the stencil holds both triangles)
      for (int j = i + 1; j < nd; j++) {
        const double m = 0.5 * (a[(size_t)i * nd + j] + a[(size_t)j * nd + i]);
        a[(size_t)i * nd + j] = a[(size_t)j * nd + i] = m;
      }
    // inverse on the device (a host inverse of 1536 unknowns took 0.2-0.4 s)
    DevBuf dm, dp;
    PZG_TRY(dev_upload(dm, a.data(), a.size(), c.stream));
    if (int rc = dev_alloc(dp, sizeof(double) * 2 * nd + 64)) {
      dev_free(dm);
      return rc;
    }
    double *prow = dp.as<double>(), *pcol = prow + nd;
    int *fail = reinterpret_cast<int *>(pcol + nd);
    PZG_HIP(hipMemsetAsync(fail, 0, sizeof(int), c.stream));
    const int64_t nn2 = (int64_t)nd * nd;
    for (int k = 0; k < nd; k++) {
      hipLaunchKernelGGL(k_gj_save, dim3((nd + TPB - 1) / TPB), dim3(TPB), 0, c.stream, nd, dm.as<double>(), k,
                         prow, pcol);
      hipLaunchKernelGGL(k_gj_step, dim3((unsigned)((nn2 + TPB - 1) / TPB)), dim3(TPB), 0, c.stream, nd,
                         dm.as<double>(), k, (const double *)prow, (const double *)pcol, fail);
    }
    PZG_TRY(dev_alloc(c.d_mg_cinv, sizeof(float) * nn2));
    hipLaunchKernelGGL(k_d2f_n, dim3((unsigned)((nn2 + TPB - 1) / TPB)), dim3(TPB), 0, c.stream, nn2,
                       dm.as<double>(), c.d_mg_cinv.as<float>());
    PZG_HIP(hipGetLastError());
    int hf = 0;
    PZG_HIP(hipMemcpyAsync(&hf, fail, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    dev_free(dm);
    dev_free(dp);
    if (hf) {
      set_error("multigrid preconditioner: the coarsest operator is not positive definite");
      return PZG_EUNSUP;
    }
    c.mg_ncoarse = nd;
  }
  // largest eigenvalues of M^-1 A: level 0, then every smoothed lattice level
  {
    if (c.mg_les) PZG_TRY(les_prepare(c));  // the learned smoother of the current assembly
    auto op = [&](const float *x, float *y) { return op0(c, x, y, nullptr, false); };
    PZG_TRY(lanczos_lmax<BS>(c, c.nb, c.d_bjinv.as<float>(), (int64_t)BS * BS, 1, c.d_mg_r0.as<float>(),
                             c.d_mg_d0.as<float>(), c.d_mg_t0.as<float>(), c.d_mg_w0.as<float>(), op,
                             c.mg_lmax0, c.mg_les));
  }
  for (size_t k = 0; k + (dense ? 1 : 0) < nl; k++) {
    MgLevel &l = c.mg[k];
    auto op = [&](const float *x, float *y) { return op_lattice<BS>(c, l, x, y, nullptr); };
    PZG_TRY(lanczos_lmax<BS>(c, l.nn, l.minv.as<float>(), 1, l.nn, l.x.as<float>(), l.b.as<float>(),
                             l.d.as<float>(), l.t.as<float>(), op, l.lmax));
  }
  PZG_HIP(hipStreamSynchronize(c.stream));
  c.mg_ready = true;
  return PZG_OK;
}

// z = V-cycle applied to r; then p = z (when given) and the z.q partials
// (when q is given), as the block-Jacobi update leaves them
template <int BS>
int apply_impl(Ctx &c, const float *r, float *z, float *p, const float *q, SolveScalars *sc,
               double *partials) {
  const LevelView L0 = view0(c);
  auto op_0 = [&](const float *x, float *y, bool ps) { return op0(c, x, y, sc, ps); };
  const int nl = (int)mg_levels(c);
  const bool dense = mg_dense_coarse(c);
  std::vector<LevelView> V(nl);
  for (int k = 0; k < nl; k++) V[k] = view_l(c, c.mg[k]);
  // first level of the tail (nl: none)
  int kt = nl;
  if (dense) {
    int64_t fl = 0;
    while (kt > 0 && nl - (kt - 1) <= MG_TAIL_MAX) {
      const MgLevel &l = c.mg[kt - 1];
      const int64_t by = l.nn * BS * BS * 4 * (l.n[2] == 1 ? 9 : 27), f = 3 * l.nn * BS;
      // (the coarsest level is read as its inverse, not as a stencil)
      if ((kt < nl ? by > MG_TAIL_BYTES : c.mg_ncoarse * c.mg_ncoarse * 4 > MG_TAIL_BYTES) ||
          (fl + f) * 4 > MG_TAIL_LDS)
        break;
      fl += f;
      kt--;
    }
    if (nl - kt < 2) kt = nl;  // the dense solve alone is a launch either way
  }
  auto first = [&](int k) { return k < nl - 1 || !dense ? V[k].m : (const float *)nullptr; };  // smoothed levels
  PZG_TRY(smooth_pre<BS>(c, L0, r, z, op_0, sc));
  hipLaunchKernelGGL(k_restrict0<BS>, dim3(grid1(c.mg[0].nn)), dim3(TPB), 0, c.stream, c.mg[0].nn,
                     c.d_mg_vmap.as<int32_t>(), c.d_mg_dsq.as<float>(), L0.r, L0.t, c.mg[0].b.as<float>(), first(0),
                     V[0].ch.c0, c.mg[0].d.as<float>(), sc);
  PZG_HIP(hipGetLastError());
  for (int k = 0; k + 1 < nl && k < kt; k++) {
    MgLevel &l = c.mg[k], &q = c.mg[k + 1];
    hipLaunchKernelGGL(k_lat_res<BS>, dim3(grid1(l.nn), BS), dim3(TPB), 0, c.stream, dims_of(l), l.nn,
                       l.A.as<float>(), l.b.as<float>(), l.d.as<float>(), l.r.as<float>(), sc);
    hipLaunchKernelGGL(k_lat_restrict<BS>, dim3(grid1(q.nn)), dim3(TPB), 0, c.stream, dims_of(q), dims_of(l),
                       l.r.as<float>(), q.b.as<float>(), first(k + 1), V[k + 1].ch.c0, q.d.as<float>(), sc);
    PZG_HIP(hipGetLastError());
  }
  if (kt < nl) {
    TailArgs t;
    std::memset(&t, 0, sizeof(t));
    t.nl = nl - kt;
    int off = 0;
    for (int k = kt; k < nl; k++) {
      const MgLevel &l = c.mg[k];
      for (int d = 0; d < 3; d++) t.n[k - kt][d] = l.n[d];
      t.off[k - kt] = off;
      off += (int)(3 * l.nn * BS);
      t.A[k - kt] = l.A.as<float>();
      t.m[k - kt] = l.minv.as<float>();
      t.c0[k - kt] = V[k].ch.c0;
    }
    t.cinv = c.d_mg_cinv.as<float>();
    t.b = c.mg[kt].b.as<float>();
    t.d = c.mg[kt].d.as<float>();
    t.x = c.mg[kt].x.as<float>();
    hipLaunchKernelGGL(k_lat_tail<BS>, dim3(1), dim3(MG_TAIL_TPB), sizeof(float) * off, c.stream, t, sc);
    PZG_HIP(hipGetLastError());
  } else if (dense) {
    hipLaunchKernelGGL(k_dense, dim3(gridx(c.mg_ncoarse * 64)), dim3(TPB), 0, c.stream, (int)c.mg_ncoarse,
                       c.d_mg_cinv.as<float>(), c.mg[nl - 1].b.as<float>(), c.mg[nl - 1].x.as<float>(), sc);
    PZG_HIP(hipGetLastError());
  } else {  // x = q(M^-1 A) M^-1 b, a Chebyshev iteration from zero
    MgLevel &l = c.mg[nl - 1];
    LevelView W = V[nl - 1];
    W.ch = cheb_coeffs(l.lmax, MG_COARSE_RANGE, MG_COARSE_DEGREE);
    auto op = [&](const float *x, float *y, bool) { return op_lattice<BS>(c, l, x, y, sc); };
    PZG_TRY(smooth_pre<BS>(c, W, l.b.as<float>(), l.x.as<float>(), op, sc));
  }
  const int kup = std::min(nl - 1, kt);  // levels above the one just solved
  for (int k = kup - 1; k >= 0; k--) {
    MgLevel &l = c.mg[k], &q = c.mg[k + 1];
    const bool plane = l.n[2] == 1;
    if (!plane)
      hipLaunchKernelGGL(k_lat_prolong<BS>, dim3(grid1(l.nn * BS)), dim3(TPB), 0, c.stream, dims_of(q), dims_of(l),
                         q.x.as<float>(), l.d.as<float>(), sc);
    constexpr int NT = lat_nt<BS>();
    hipLaunchKernelGGL(k_lat_post<BS>, dim3((unsigned)std::max<int64_t>(1, (l.nn + NT - 1) / NT)), dim3(NT * BS), 0,
                       c.stream, dims_of(l), l.nn, l.A.as<float>(), l.minv.as<float>(), l.b.as<float>(),
                       l.d.as<float>(), dims_of(q), plane ? q.x.as<float>() : (const float *)nullptr, V[k].ch.c0,
                       l.x.as<float>(), k == 0 ? c.d_mg_vmap.as<int32_t>() : (const int32_t *)nullptr,
                       c.d_mg_dsq.as<float>(), z, sc);
    PZG_HIP(hipGetLastError());
  }
  if (kup == 0) {
    hipLaunchKernelGGL(k_prolong0<BS>, dim3(grid1(c.mg[0].nn)), dim3(TPB), 0, c.stream, c.mg[0].nn,
                       c.d_mg_vmap.as<int32_t>(), c.d_mg_dsq.as<float>(), c.mg[0].x.as<float>(), z, sc);
    PZG_HIP(hipGetLastError());
  }
  PZG_TRY(smooth_post<BS>(c, L0, r, z, op_0, sc));
  // the learned path leaves the penalty rows to the FP64 refinement
  if ((p || q) && c.mg_les) PZG_TRY(pen_zero32(c, z));
  if (p || q) {
    // same grid as the FCG update kernel, whose partials slot 1 this replaces
    hipLaunchKernelGGL(k_mg_finish<BS>, dim3(gridr(c.nb)), dim3(TPB), 0, c.stream, c.nb, z, p, q, sc, partials);
    PZG_HIP(hipGetLastError());
  }
  return PZG_OK;
}

}  // namespace

void mg_free(Ctx &c) {
  pen_free(c);
  for (MgLevel &l : c.mg)
    for (DevBuf *b : {&l.A, &l.minv, &l.x, &l.b, &l.r, &l.d, &l.t}) dev_free(*b);
  c.mg.clear();
  c.mg_struct = false;
  for (DevBuf *b : {&c.d_mg_vmap, &c.d_mg_vinv, &c.d_mg_dsq, &c.d_mg_cinv, &c.d_mg_r0, &c.d_mg_d0, &c.d_mg_t0, &c.d_mg_w0,
                    &c.d_mg_lz})
    dev_free(*b);
  c.mg_ready = false;
}

int mg_setup(Ctx &c, bool use_mf, bool ext) {
  c.mg_ready = false;
  c.mg_use_mf = use_mf;
  c.mg_ext = ext;
  if (c.mg_degree < 1 || c.mg_degree > 8 || !(c.mg_range > 1.)) {
    set_error("multigrid preconditioner: degree must be 1..8 and the range above 1");
    return PZG_EINVAL;
  }
  if (c.bs == 3) return setup_impl<3>(c);
  if (c.bs == 1) return setup_impl<1>(c);
  set_error("multigrid preconditioner: nstate must be 1 or 3");
  return PZG_EUNSUP;
}

int mg_apply(Ctx &c, const float *r, float *z, float *p, const float *q, SolveScalars *sc, double *partials) {
  if (!c.mg_ready) {
    set_error("multigrid preconditioner: not set up");
    return PZG_ESTATE;
  }
  if (c.bs == 3) return apply_impl<3>(c, r, z, p, q, sc, partials);
  return apply_impl<1>(c, r, z, p, q, sc, partials);
}

}  // namespace pzg
