// pzg_device.h -- device helpers shared by the solver and learned kernels:
// wavefront/block sums and the deterministic two-level reduction.
#pragma once
#include <hip/hip_runtime.h>

namespace pzg {

constexpr int RED_TPB = 256;

// Workgroups are dispatched round-robin over the XCDs (workgroup b runs on XCD
// b % NXCD), and each XCD has its own L2.  xcd_block_range gives workgroup
// blockIdx.x a contiguous slice [lo, hi) of [0, n) such that the slices of the
// workgroups of one XCD are adjacent: XCD k covers about [k n/NXCD,
// (k+1) n/NXCD), so the gathered operands of neighbouring rows stay in that
// XCD's L2.
constexpr int NXCD = 8;
__device__ inline void xcd_block_range(int64_t n, int64_t &lo, int64_t &hi) {
  const int G = (int)gridDim.x, b = (int)blockIdx.x;
  const int x = b % NXCD, i = b / NXCD;
  const int per = G / NXCD, rem = G % NXCD;
  const int64_t vb = (int64_t)x * per + (x < rem ? x : rem) + i;
  lo = n * vb / G;
  hi = n * (vb + 1) / G;
}

// The slab [lo, hi) of [0, n) owned by this workgroup's XCD, the index i of
// the workgroup among that XCD's gk workgroups.  Interleaving the XCD's
// workgroups over its slab (tile i, i + gk, ...) keeps the rows in flight on
// one XCD in a narrow band, so the gathered operands fit in its L2.
#ifndef PZG_XCD_INTERLEAVE
#define PZG_XCD_INTERLEAVE 1
#endif
__device__ inline void xcd_slab(int64_t n, int64_t &lo, int64_t &hi, int &i, int &gk) {
  const int G = (int)gridDim.x, b = (int)blockIdx.x;
  const int x = b % NXCD;
  const int per = G / NXCD, rem = G % NXCD;
  i = b / NXCD;
  gk = per + (x < rem ? 1 : 0);
  const int64_t first = (int64_t)x * per + (x < rem ? x : rem);
  lo = n * first / G;
  hi = n * (first + gk) / G;
}
constexpr int MAXBLK = 2048;  // partial-sum slots per reduction
constexpr int NSLOT = 4;

// Cross-lane moves inside a row of 16 lanes by DPP (no LDS round trip: a
// __shfl of a double is two ds_bpermute of some 60 cycles each).
template <int CTRL> __device__ inline float dpp_move(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ inline double dpp_move(double v) {
  const int64_t b = __builtin_bit_cast(int64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffff), CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (int64_t)((uint64_t)hi << 32 | lo));
}
// sum over the row of 16 lanes in each of its lanes (row_ror 8, 4, 2, 1: the
// additions of an xor butterfly)
template <class T> __device__ inline T row16_sum(T v) {
  v += dpp_move<0x128>(v);
  v += dpp_move<0x124>(v);
  v += dpp_move<0x122>(v);
  v += dpp_move<0x121>(v);
  return v;
}
__device__ inline double lane_value(double v, int lane) {
  const int64_t b = __builtin_bit_cast(int64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(b & 0xffffffff), lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, (int64_t)((uint64_t)hi << 32 | lo));
}

// sum over the wavefront (every lane active) in every lane
__device__ inline double wave_sum(double v) {
  v = row16_sum(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// Sum of v over the block; result valid in thread 0.
__device__ inline double block_sum(double v, double *sm) {
  v = wave_sum(v);
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sm[w] = v;
  __syncthreads();
  double s = 0.;
  if (threadIdx.x == 0)
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) s += sm[k];
  return s;
}

// Stores this block's sums of v into partials[k*MAXBLK + blockIdx.x] (plain
// stores: a one-block kernel that follows sums them, ordered by the kernel
// boundary).  A last-block reduction inside the producer was measured slower:
// its device-scope fence writes back every XCD's dirty L2 lines, 0.14 ms on a
// residual of 66k rows and 0.3 ms on a vector pass over 6.4M entries that
// takes 0.03 ms without it.
template <int NV>
__device__ inline void block_partials(const double (&v)[NV], double *partials) {
  __shared__ double sm[RED_TPB / 64];
  for (int k = 0; k < NV; k++) {
    double s = block_sum(v[k], sm);
    if (threadIdx.x == 0) partials[k * MAXBLK + blockIdx.x] = s;
  }
}

// Fixed-order sum of nblk partials of one slot, run by a single block;
// result valid in thread 0.
__device__ inline double sum_partials(const double *partials, int slot, int nblk) {
  __shared__ double sm[RED_TPB / 64];
  double s = 0.;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) s += partials[slot * MAXBLK + b];
  return block_sum(s, sm);
}

}  // namespace pzg
