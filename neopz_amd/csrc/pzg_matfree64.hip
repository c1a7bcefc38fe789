// pzg_matfree64.hip -- FP64 products with the assembled K on meshes of
// identical affine p = 2 hexahedra, from the coefficient-1 element matrix.
//
// On such a mesh the stored matrix is K = sum_e coef_e P_e^T K_ref P_e plus
// the penalty matrices of the Dirichlet faces (k_vol_blk and k_bc write it
// that way), so a product needs 81 x 81 doubles of K_ref, one coefficient per
// element and the vectors instead of the block CSR: 2 * 81^2 flop per element
// on the FP64 matrix cores against 76 bytes per stored block.  AddKel's drop
// rule (|coef_e K_ref(i,j)| < 1e-12 is not added) is part of K: kf_prepare
// zeroes the entries it drops for every element of the mesh and leaves the
// product to the block CSR when it would drop an entry for some elements only.
// The result differs from the block CSR's by the rounding of the sums.
//
// k_kf_elem: y_e = coef_e K_ref u_e, element-major; k_kf_rows sums the
// elements of each row in element order, adds the Dirichlet faces and finishes
// what the caller needs (no atomics: the result is deterministic).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "pzg_device.h"
#include "pzg_internal.h"

namespace pzg {

namespace {

constexpr int KF_TPB = 256;
constexpr int KF_NSH = 27;   // shapes of the p = 2 hexahedron
constexpr int KF_NWV = 8;    // wavefronts per workgroup on large meshes (64.5 KB of tables each)
constexpr int KF_NSHB = 9;   // shapes of its faces

typedef double kf_d4 __attribute__((ext_vector_type(4)));

constexpr int kf_ksteps(int ns) { return (KF_NSH + 3) / 4 * ns; }
constexpr int kf_rtiles(int ns) { return (KF_NSH * ns + 15) / 16; }

__global__ void k_kf_blk(int64_t n, const int64_t *__restrict__ vconn, const int64_t *__restrict__ aidx,
                         int32_t *__restrict__ blk) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) blk[t] = (int32_t)aidx[vconn[t]];
}

__global__ void k_kf_fill(int64_t n, int32_t v, int32_t *__restrict__ p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}
__global__ void k_kf_index(int64_t n, const int32_t *__restrict__ row, int32_t *__restrict__ pidx) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) pidx[row[t]] = (int32_t)t;
}

// big * (phi_i, phi_j) of every Dirichlet face, as k_bc integrates it (area
// element by Gram-Schmidt of the two tangents), one thread per entry
__global__ void k_kf_bm(int64_t nbcd, const int32_t *__restrict__ faces, const ElemTables *__restrict__ tab,
                        const double *__restrict__ xyz, const int64_t *__restrict__ nodes, double big,
                        double *__restrict__ bm) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nbcd * KF_NSHB * KF_NSHB) return;
  const int64_t f = t / (KF_NSHB * KF_NSHB), e = faces[f];
  const int i = (int)(t / KF_NSHB % KF_NSHB), j = (int)(t % KF_NSHB);
  double s = 0.;
  for (int q = 0; q < tab->nq; q++) {
    double a[3] = {0., 0., 0.}, b[3] = {0., 0., 0.};
    for (int k = 0; k < 4; k++) {
      const double *x = xyz + 3 * nodes[e * 4 + k];
      for (int d = 0; d < 3; d++) {
        a[d] += x[d] * tab->cdphi[q][0][k];
        b[d] += x[d] * tab->cdphi[q][1][k];
      }
    }
    const double n1 = sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
    const double d12 = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
    double n2 = 0.;
    for (int d = 0; d < 3; d++) {
      const double v = b[d] - d12 * (a[d] / n1) / n1;
      n2 += v * v;
    }
    s += tab->phi[q][i] * tab->phi[q][j] * (tab->w[q] * fabs(n1 * sqrt(n2)));
  }
  const double v = big * s;
  bm[t] = fabs(v) < 1.e-12 ? 0. : v;
}

// y_e = coef_e K_ref u_e on the FP64 matrix cores: K_ref is the A operand
// (rows in tiles of 16, staged in LDS in operand order), 16 elements the
// columns of B, one tile of elements per wavefront and pass.  RT row tiles per
// wavefront: all of them on large meshes (each u_e is gathered once), a third
// (blockIdx.y picks it) where the element tiles alone would leave SIMDs idle.
// Operand layouts of the 16x16x4 instruction (wave64): A: lane l holds
// A[l%16][l/16]; B: lane l holds B[l/16][l%16]; D: lane l, component r holds
// D[l/16 + 4r][l%16].
// Bound by the FP64 matrix cores: 126 instructions of 64 cycles per 16 elements
// (81 padded to 96 x 84), 54 us for 64^3 elements at the peak rate.  Measured
// with k_kf_rows, us per product against the block CSR product it replaces:
// 64^3 115 + 116 (2100 to 2770: 10.4 GB streamed), 48^3 60 + 40 (1010),
// 24^3 15 + 9 (134), 6^3 9 + 5.
// k order: step t = NS*s4 + c holds component c of the shapes 4*s4 + (0..3), so
// a lane gathers one block index per NS steps and its values are contiguous.
// The A reads of a step stay behind the step before it (sched_barrier): hoisted
// together they spilled the accumulators.
template <int NS, int RT, int NWV>
__global__ __launch_bounds__(NWV * 64) void k_kf_elem(int64_t nvol, const double *__restrict__ tab,
                                                      const int32_t *__restrict__ blk,
                                                      const double *__restrict__ x,
                                                      const double *__restrict__ coefv, double coef0,
                                                      double *__restrict__ ye, const SolveScalars *sc) {
  if (sc && sc->done) return;
  constexpr int NE = KF_NSH * NS, TK = kf_ksteps(NS), S4 = (KF_NSH + 3) / 4;
  __shared__ double sA[RT * TK * 64];
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l >> 4;
  {
    const double *src = tab + (int64_t)blockIdx.y * (RT * TK * 64);
    for (int t = tid; t < RT * TK * 64; t += NWV * 64) sA[t] = src[t];
  }
  __syncthreads();
  const int row0 = blockIdx.y * RT * 16;
  int64_t lo, hi;
  int xi, xg;
  xcd_slab((nvol + 15) / 16, lo, hi, xi, xg);
  for (int64_t tile = lo + (int64_t)xi * NWV + wv; tile < hi; tile += (int64_t)xg * NWV) {
    const int64_t e = tile * 16 + (l & 15);
    const bool ok = e < nvol;
    const int64_t ec = ok ? e : 0;
    // branch-free gathers (clamped addresses): every index, then every value
    int32_t bb[S4];
#pragma unroll
    for (int s = 0; s < S4; s++) {
      const int sh = 4 * s + lr;
      bb[s] = blk[ec * KF_NSH + (sh < KF_NSH ? sh : KF_NSH - 1)];
    }
    double u[S4][NS];
#pragma unroll
    for (int s = 0; s < S4; s++)
#pragma unroll
      for (int c = 0; c < NS; c++) u[s][c] = x[(int64_t)bb[s] * NS + c];
    const double cf = coefv ? coefv[ec] : coef0;
    if (4 * (S4 - 1) + lr >= KF_NSH)  // the shape past the last one
#pragma unroll
      for (int c = 0; c < NS; c++) u[S4 - 1][c] = 0.;
    kf_d4 acc[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) acc[r] = kf_d4{0., 0., 0., 0.};
#pragma unroll
    for (int s = 0; s < S4; s++)
#pragma unroll
      for (int c = 0; c < NS; c++) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RT; r++)
          acc[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(sA[(r * TK + NS * s + c) * 64 + l], u[s][c], acc[r], 0, 0, 0);
      }
    if (ok) {
      double *o = ye + e * NE;
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int row = row0 + 16 * r + lr + 4 * i;
          if (row < NE) o[row] = cf * acc[r][i];
        }
    }
  }
}

// Row sums of the element products, one thread per equation, plus the
// Dirichlet faces of the row.  MODE 0: out = alpha (K x) + beta y; 1: out =
// K x with the partials of x.(K x) in slot 0; 2: out (if given) = f - K x with
// |out|^2 and |f|^2 in slots 0 and 1.
template <int NS, int MODE>
__global__ __launch_bounds__(KF_TPB) void k_kf_rows(int64_t neq, const int64_t *__restrict__ iptr,
                                                    const int32_t *__restrict__ inc,
                                                    const double *__restrict__ ye,
                                                    const int32_t *__restrict__ pidx,
                                                    const int32_t *__restrict__ pptr,
                                                    const int32_t *__restrict__ psrc,
                                                    const int32_t *__restrict__ bblk,
                                                    const double *__restrict__ bm,
                                                    const double *__restrict__ x,
                                                    const double *__restrict__ f, double alpha, double beta,
                                                    double *__restrict__ out, const SolveScalars *sc,
                                                    double *partials) {
  if (sc && sc->done) return;
  constexpr int NE = KF_NSH * NS, MAXI = 8;
  double s0 = 0., s1 = 0.;
  int64_t lo, hi;
  int xi, xg;
  xcd_slab(neq, lo, hi, xi, xg);
  for (int64_t i = lo + (int64_t)xi * KF_TPB + threadIdx.x; i < hi; i += (int64_t)xg * KF_TPB) {
    const int64_t A = i / NS;
    const int k = (int)(i - A * NS);
    const int64_t b0 = iptr[A];
    const int m = (int)(iptr[A + 1] - b0);  // <= MAXI (checked where the lists are built)
    const int32_t pr = pidx ? pidx[A] : -1;
    const double xv = MODE == 1 ? x[i] : MODE == 2 ? f[i] : f ? f[i] : 0.;
    int32_t v[MAXI];
#pragma unroll
    for (int j = 0; j < MAXI; j++) v[j] = inc[b0 + (j < m ? j : 0)];
    double y[MAXI];
#pragma unroll
    for (int j = 0; j < MAXI; j++) y[j] = ye[(int64_t)(v[j] >> 5) * NE + (v[j] & 31) * NS + k];
    double s = 0.;
#pragma unroll
    for (int j = 0; j < MAXI; j++)
      if (j < m) s += y[j];
    if (pr >= 0)
      for (int32_t q = pptr[pr]; q < pptr[pr + 1]; q++) {
        const int32_t slot = psrc[q];
        const double *mr = bm + (int64_t)slot * KF_NSHB;
        const int32_t *bj = bblk + slot / KF_NSHB * KF_NSHB;
        for (int j = 0; j < KF_NSHB; j++) s += mr[j] * x[(int64_t)bj[j] * NS + k];
      }
    if (MODE == 0) {
      out[i] = alpha * s + (f ? beta * xv : 0.);
    } else if (MODE == 1) {
      out[i] = s;
      s0 += s * xv;
    } else {
      const double r = xv - s;
      if (out) out[i] = r;
      s0 += r * r;
      s1 += xv * xv;
    }
  }
  if (MODE == 1) {
    double vv[1] = {s0};
    block_partials<1>(vv, partials);
  } else if (MODE == 2) {
    double vv[2] = {s0, s1};
    block_partials<2>(vv, partials);
  }
}

// mesh-level part: element blocks, output buffer, Dirichlet faces by row
int kf_setup(Ctx &c) {
  if (c.kf_struct) return PZG_OK;
  hipStream_t s = c.stream;
  const int64_t n = c.nvol * KF_NSH;
  PZG_TRY(dev_alloc(c.d_kf_blk, sizeof(int32_t) * n));
  hipLaunchKernelGGL(k_kf_blk, dim3((unsigned)((n + KF_TPB - 1) / KF_TPB)), dim3(KF_TPB), 0, s, n,
                     c.d_vconn.as<int64_t>(), c.d_aidx.as<int64_t>(), c.d_kf_blk.as<int32_t>());
  PZG_TRY(dev_alloc(c.d_kf_ye, sizeof(double) * n * c.nstate));
  std::vector<int32_t> faces, bblk;
  std::vector<int64_t> key;  // (block row, slot)
  for (int64_t e = 0; e < c.nbc; e++) {
    if (c.bc_type[c.bc_id[e]] != PZG_BC_DIRICHLET) continue;
    for (int i = 0; i < KF_NSHB; i++) {
      const int64_t b = c.aidx[c.bc_conn[e * c.bc_nsides + c.tbc.shape_side[i]]];
      key.push_back((b << 32) | (int64_t)bblk.size());
      bblk.push_back((int32_t)b);
    }
    faces.push_back((int32_t)e);
  }
  c.kf_nface = (int64_t)faces.size();
  if (c.kf_nface) {
    std::sort(key.begin(), key.end());
    std::vector<int32_t> row, ptr, src;
    for (int64_t k : key) {
      const int32_t b = (int32_t)(k >> 32);
      if (row.empty() || row.back() != b) {
        row.push_back(b);
        ptr.push_back((int32_t)src.size());
      }
      src.push_back((int32_t)(k & 0x7fffffff));
    }
    ptr.push_back((int32_t)src.size());
    DevBuf d_faces, d_row;
    int rc = dev_upload(d_faces, faces.data(), faces.size(), s);
    if (rc == PZG_OK) rc = dev_upload(d_row, row.data(), row.size(), s);
    if (rc == PZG_OK) rc = dev_upload(c.d_kf_bblk, bblk.data(), bblk.size(), s);
    if (rc == PZG_OK) rc = dev_upload(c.d_kf_pptr, ptr.data(), ptr.size(), s);
    if (rc == PZG_OK) rc = dev_upload(c.d_kf_psrc, src.data(), src.size(), s);
    const int64_t nm = c.kf_nface * KF_NSHB * KF_NSHB;
    if (rc == PZG_OK) rc = dev_alloc(c.d_kf_bm, sizeof(double) * nm);
    if (rc == PZG_OK) rc = dev_alloc(c.d_kf_pidx, sizeof(int32_t) * c.nb);
    if (rc == PZG_OK) {
      const int64_t nr = (int64_t)row.size();
      hipLaunchKernelGGL(k_kf_bm, dim3((unsigned)((nm + KF_TPB - 1) / KF_TPB)), dim3(KF_TPB), 0, s, c.kf_nface,
                         d_faces.as<int32_t>(), c.d_tbc.as<ElemTables>(), c.d_xyz.as<double>(),
                         c.d_bnodes.as<int64_t>(), c.big, c.d_kf_bm.as<double>());
      hipLaunchKernelGGL(k_kf_fill, dim3((unsigned)((c.nb + KF_TPB - 1) / KF_TPB)), dim3(KF_TPB), 0, s, c.nb, -1,
                         c.d_kf_pidx.as<int32_t>());
      hipLaunchKernelGGL(k_kf_index, dim3((unsigned)((nr + KF_TPB - 1) / KF_TPB)), dim3(KF_TPB), 0, s, nr,
                         d_row.as<int32_t>(), c.d_kf_pidx.as<int32_t>());
      if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
        set_error("FP64 element products: set-up kernels failed");
        rc = PZG_EHIP;
      }
    }
    dev_free(d_faces);
    dev_free(d_row);
    PZG_TRY(rc);
  }
  c.kf_struct = true;
  c.kf_ndrop = -1;
  return PZG_OK;
}

// K_ref in operand order with the entries that AddKel drops for every element
// zeroed; *ok false when it would drop an entry for some elements only
int kf_coef(Ctx &c, bool *ok) {
  *ok = false;
  double lo = HUGE_VAL, hi = 0.;
  if (c.vol_coef.empty()) {
    lo = hi = std::fabs(c.material == PZG_MAT_ELAST3D ? c.E : c.scale);
  } else {
    for (int64_t e = 0; e < c.nvol; e++) {
      const double a = std::fabs(c.vol_coef[e]);
      if (!(a < HUGE_VAL)) return PZG_OK;  // infinite or not a number
      if (a > 0.) lo = std::min(lo, a);    // (a zero coefficient adds nothing either way)
      hi = std::max(hi, a);
    }
  }
  if (!(hi > 0.) || !(hi < HUGE_VAL)) return PZG_OK;
  const int NE = KF_NSH * c.nstate, TK = kf_ksteps(c.nstate), R = kf_rtiles(c.nstate);
  int64_t nd = 0;
  for (double v : c.blk_kref) {
    const double a = std::fabs(v);
    if (a * hi < 0.999999e-12) nd++;  // dropped by every element
    else if (!(a * lo >= 1.000001e-12)) return PZG_OK;
  }
  if (nd != c.kf_ndrop) {  // (the dropped entries are the nd smallest: the same set as before)
    std::vector<double> t((size_t)R * TK * 64, 0.);
    for (int r = 0; r < R; r++)
      for (int k = 0; k < TK; k++)
        for (int l = 0; l < 64; l++) {
          const int i = 16 * r + l % 16, sh = 4 * (k / c.nstate) + l / 16, j = sh * c.nstate + k % c.nstate;
          if (i >= NE || sh >= KF_NSH) continue;
          const double v = c.blk_kref[(size_t)i * NE + j];
          if (!(std::fabs(v) * hi < 0.999999e-12)) t[((size_t)r * TK + k) * 64 + l] = v;
        }
    PZG_TRY(dev_upload(c.d_kf_tab, t.data(), t.size(), c.stream));
    PZG_HIP(hipStreamSynchronize(c.stream));
    c.kf_ndrop = nd;
  }
  *ok = true;
  return PZG_OK;
}

template <int NS>
void launch_elem(Ctx &c, const double *x, const SolveScalars *sc) {
  const int64_t tiles = (c.nvol + 15) / 16;
  const double *coef = c.vol_coef.empty() ? nullptr : c.d_vcoef.as<double>();
  const double coef0 = c.material == PZG_MAT_ELAST3D ? c.E : c.scale;
  auto grid8 = [](int64_t g) { return (unsigned)((std::max<int64_t>(g, 1) + 7) / 8 * 8); };
  if (NS == 3 && tiles < KF_SPLIT_TILES) {
    const dim3 g(grid8((tiles + 3) / 4), 3);
    hipLaunchKernelGGL((k_kf_elem<NS, NS == 3 ? 2 : kf_rtiles(NS), 4>), g, dim3(256), 0, c.stream, c.nvol,
                       c.d_kf_tab.as<double>(), c.d_kf_blk.as<int32_t>(), x, coef, coef0, c.d_kf_ye.as<double>(), sc);
  } else {
    const dim3 g(grid8(std::min<int64_t>((tiles + KF_NWV - 1) / KF_NWV, 512)));  // two workgroups per CU
    hipLaunchKernelGGL((k_kf_elem<NS, kf_rtiles(NS), KF_NWV>), g, dim3(KF_NWV * 64), 0, c.stream, c.nvol,
                       c.d_kf_tab.as<double>(), c.d_kf_blk.as<int32_t>(), x, coef, coef0, c.d_kf_ye.as<double>(), sc);
  }
}

}  // namespace

bool kf_usable_mesh(const Ctx &c) {
  return c.has_mesh && c.has_struct && !c.external_csr && !c.has_dep && !c.filt && c.blk_asm && c.aff_on &&
         c.blk_full && c.bc_mf_ok && c.vol_rules.size() == 1 && c.bc_rules.size() <= 1 && c.dim == 3 &&
         c.tvol.nsh == KF_NSH && (c.nbc == 0 || (c.tbc.nsh == KF_NSHB && c.bc_ncorner == 4)) && c.bs == c.nstate &&
         c.nvol * KF_NSH < INT32_MAX && c.nbc * KF_NSHB < INT32_MAX && c.nb < INT32_MAX;
}
int kf_setup_mesh(Ctx &c) { return kf_setup(c); }

// The products below stand for those of the block CSR on this system
bool kf_usable(const Ctx &c) {
  return kf_usable_mesh(c) && c.assembled && !c.kel_added && c.nvol >= (c.nstate == 3 ? KF_MIN_EL3 : KF_MIN_EL1);
}

int kf_prepare(Ctx &c, bool *ok) {
  *ok = c.kf_valid;
  if (c.kf_valid || !kf_usable(c)) return PZG_OK;
  PZG_TRY(kf_setup(c));
  PZG_TRY(kf_coef(c, ok));
  c.kf_valid = *ok;
  return PZG_OK;
}

// Every buffer, value and choice that kf_apply puts into its launches.
void kf_key(const Ctx &c, std::vector<uint64_t> &key) {
  key_add(key, c.bs, c.neq, c.nvol, c.kf_nface, c.vol_coef.empty(), c.material == PZG_MAT_ELAST3D ? c.E : c.scale,
          c.d_vcoef, c.d_kf_tab, c.d_kf_blk, c.d_kf_ye, c.d_blk_iptr, c.d_blk_inc, c.d_kf_pidx, c.d_kf_pptr,
          c.d_kf_psrc, c.d_kf_bblk, c.d_kf_bm);
}

int kf_rows_grid(const Ctx &c) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((c.neq + KF_TPB - 1) / KF_TPB, MAXBLK));
}

int kf_apply(Ctx &c, int mode, const double *x, const double *f, double alpha, double beta, double *out,
             const SolveScalars *sc, double *partials) {
  if (!c.kf_valid) {
    set_error("FP64 element products: not prepared");
    return PZG_ESTATE;
  }
  if (c.bs == 3) launch_elem<3>(c, x, sc);
  else launch_elem<1>(c, x, sc);
  const dim3 g(kf_rows_grid(c));
  const int32_t *pidx = c.kf_nface ? c.d_kf_pidx.as<int32_t>() : nullptr;
#define KF_ROWS(NS, MODE)                                                                                           \
  hipLaunchKernelGGL((k_kf_rows<NS, MODE>), g, dim3(KF_TPB), 0, c.stream, c.neq, c.d_blk_iptr.as<int64_t>(),       \
                     c.d_blk_inc.as<int32_t>(), c.d_kf_ye.as<double>(), pidx, c.d_kf_pptr.as<int32_t>(),           \
                     c.d_kf_psrc.as<int32_t>(), c.d_kf_bblk.as<int32_t>(), c.d_kf_bm.as<double>(), x, f, alpha,    \
                     beta, out, sc, partials)
  if (c.bs == 3) {
    if (mode == KF_AXPBY) KF_ROWS(3, 0);
    else if (mode == KF_DOT) KF_ROWS(3, 1);
    else KF_ROWS(3, 2);
  } else {
    if (mode == KF_AXPBY) KF_ROWS(1, 0);
    else if (mode == KF_DOT) KF_ROWS(1, 1);
    else KF_ROWS(1, 2);
  }
#undef KF_ROWS
  PZG_HIP(hipGetLastError());
  return PZG_OK;
}

}  // namespace pzg
