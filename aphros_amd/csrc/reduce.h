// Deterministic reductions for the aphpois kernels.
//
// A reducing kernel calls block_partial(): every workgroup reduces its values
// (sum, or max for the slots flagged in MaxMask) with a fixed wave64 butterfly
// and a fixed cross-wave order and writes them to partials[k * nblk + lb] with
// plain stores.  A one-workgroup-per-system finalize kernel then calls
// reduce_partials(), which sums the partials in block order; the kernel
// boundary makes the partials visible, so no fences or atomics are needed and
// the total does not depend on scheduling.
#pragma once

#include "common.h"

namespace aph {

// x of another lane by a DPP control (within rows of 16 lanes)
template <int Ctrl>
__device__ __forceinline__ double dpp_of(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, Ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), Ctrl, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// x of a given lane, uniform
__device__ __forceinline__ double lane_of(double x, int lane) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Sum (or max) over the wavefront, the same in every lane: within rows of 16
// lanes by DPP moves (neighbour, pair, half-row mirror, row mirror), then over
// the four rows.  Every lane must take part.  (A butterfly of __shfl_xor goes
// through LDS twelve times: ~0.25 us against ~0.05 us.)
template <int NV, unsigned MaxMask>
__device__ __forceinline__ void wave_reduce(double (&v)[NV]) {
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const bool mx = (MaxMask >> k) & 1u;
    auto op = [mx](double a, double b) { return mx ? fmax(a, b) : a + b; };
    double x = v[k];
    x = op(x, dpp_of<0xB1>(x));   // quad_perm 1 0 3 2
    x = op(x, dpp_of<0x4E>(x));   // quad_perm 2 3 0 1
    x = op(x, dpp_of<0x141>(x));  // row_half_mirror
    x = op(x, dpp_of<0x140>(x));  // row_mirror
    v[k] = op(op(lane_of(x, 0), lane_of(x, 16)), op(lane_of(x, 32), lane_of(x, 48)));
  }
}

// Block-wide reduction over NT threads; the result is valid in every thread.
template <int NV, unsigned MaxMask, int NT = kBlock>
__device__ __forceinline__ void block_reduce(double (&v)[NV]) {
  __shared__ double red[NV][NT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  wave_reduce<NV, MaxMask>(v);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) red[k][wave] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double t = red[k][0];
    for (int w = 1; w < NT / 64; ++w) {
      t = ((MaxMask >> k) & 1u) ? fmax(t, red[k][w]) : t + red[k][w];
    }
    v[k] = t;
  }
  __syncthreads();
}

// Writes this workgroup's partial values.  Must be reached by every thread.
template <int NV, unsigned MaxMask, int NT = kBlock>
__device__ __forceinline__ void block_partial(double (&v)[NV], double* partials, int nblk,
                                              int lb) {
  block_reduce<NV, MaxMask, NT>(v);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) partials[(long long)k * nblk + lb] = v[k];
  }
}

// Sums (or maxes) the partials of nblk workgroups in block order; result in
// every thread of the calling workgroup.
template <int NV, unsigned MaxMask, int NT = kBlock>
__device__ __forceinline__ void reduce_partials(double (&v)[NV], const double* partials,
                                                int nblk) {
  // J independent accumulators per value (all of their loads in flight; two of
  // four values, for the registers), combined in a fixed order
  constexpr int J = NV > 3 ? 2 : 4;
  double t[NV][4] = {};
  auto add = [&](int j, int i) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const double pv = partials[(long long)k * nblk + i];
      t[k][j] = ((MaxMask >> k) & 1u) ? fmax(t[k][j], pv) : t[k][j] + pv;
    }
  };
  int i = threadIdx.x;
#pragma unroll 1
  for (; i + (J - 1) * NT < nblk; i += J * NT) {
#pragma unroll
    for (int j = 0; j < J; ++j) add(j, i + j * NT);
  }
  if (i < nblk) add(0, i);
  if (J > 2 && i + NT < nblk) add(1, i + NT);
  if (J > 2 && i + 2 * NT < nblk) add(2, i + 2 * NT);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double* s = t[k];
    v[k] = ((MaxMask >> k) & 1u) ? fmax(fmax(s[0], s[1]), fmax(s[2], s[3]))
                                 : (s[0] + s[1]) + (s[2] + s[3]);
  }
  block_reduce<NV, MaxMask, NT>(v);
}

}  // namespace aph
