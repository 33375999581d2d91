// Device helpers shared by the sparse kernels (SpMV, PCG, learned preconditioner): value indexing of
// the block layouts, wavefront / workgroup reductions and the node-block row product.
#pragma once

#include "fe_internal.h"

namespace fe_sparse {

constexpr int kBlock = 256;

// Value index of entry k (= di*D + dj) of block q.
template <int D, int LAYOUT>
__device__ __host__ inline int64_t vix(int64_t q, int k, int64_t nnzb) {
  return LAYOUT == FE_LAYOUT_PLANES ? (int64_t)k * nnzb + q : q * D * D + k;
}

// --------------------------------------------------------------------------------------------------
// reductions
// --------------------------------------------------------------------------------------------------
// Sum over the wavefront, in every lane: the butterfly over lane distances 32, 16, 8, 4, 2, 1.  The exchanges
// are register moves (swaps of half wavefronts and of rows, then lane permutations inside a row of 16):
// six dependent LDS permutes took 0.35 us, on the critical path of every reduction.  Once two
// distances have been added, all lanes they connect hold the same bits, so a rotation by 8 and by
// 4 lanes within the row of 16 meets a lane with the value the butterfly's partner holds.
template <int CTRL>
__device__ inline double dpp_move(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int CTRL>
__device__ inline float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

__device__ inline double wave_sum(double v) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  long long b = __double_as_longlong(v);
  u2 l = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
  u2 h = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  v = __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
  b = __double_as_longlong(v);
  l = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
  h = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  v = __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
  v += dpp_move<0x128>(v);  // row_ror:8
  v += dpp_move<0x124>(v);  // row_ror:4
  v += dpp_move<0x4e>(v);   // quad_perm [2,3,0,1]
  return v + dpp_move<0xb1>(v);  // quad_perm [1,0,3,2]
}

// Sum over the aligned group of G lanes (2, 4, 8 or 16) that share a row, in every lane, over the lane
// distances 1, 2, 4, 8: from 4 on a mirror image meets a lane of the other half, and all of a half's lanes
// hold its sum.
template <int G, typename T>
__device__ inline T group_sum(T v) {
  static_assert(G == 2 || G == 4 || G == 8 || G == 16, "lanes of one row of 16");
  v += dpp_move<0xb1>(v);
  if constexpr (G >= 4) v += dpp_move<0x4e>(v);
  if constexpr (G >= 8) v += dpp_move<0x141>(v);   // row_half_mirror
  if constexpr (G >= 16) v += dpp_move<0x140>(v);  // row_mirror
  return v;
}

// Lane J's value of the group of G lanes, for the lanes 0..3 of the group (J < 4).
template <int G, int J, typename T>
__device__ inline T group_lane(T v) {
  static_assert(J < G && J < 4, "a lane of the group's first four");
  constexpr int kCtrl = G == 2 ? (J | J << 2 | (2 + J) << 4 | (2 + J) << 6) : (J | J << 2 | J << 4 | J << 6);
  return dpp_move<kCtrl>(v);
}

// Sum NV values over the workgroup; result valid in thread 0.
template <int NV>
__device__ inline void block_sum(double (&v)[NV]) {
  __shared__ double red[NV][kBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) red[k][wid] = v[k];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
      for (int w = 0; w < kBlock / 64; ++w) s += red[k][w];
      v[k] = s;
    }
  __syncthreads();
}

// --------------------------------------------------------------------------------------------------
// SpMV on node-block rows.  G lanes per block row; each lane walks the row's blocks with stride G.
// --------------------------------------------------------------------------------------------------
template <typename T, int D, int G, int LAYOUT>
__device__ inline void bsr_row(const int32_t* __restrict__ bptr, const int32_t* __restrict__ bcol,
                               const T* __restrict__ vals, int64_t nnzb, const T* __restrict__ x,
                               int64_t i, int lane, T (&acc)[D]) {
#pragma unroll
  for (int d = 0; d < D; ++d) acc[d] = T(0);
  const int32_t s = bptr[i], e = bptr[i + 1];
  for (int32_t q = s + lane; q < e; q += G) {
    const int64_t j = bcol[q];
    T xj[D];
#pragma unroll
    for (int d = 0; d < D; ++d) xj[d] = x[j * D + d];
#pragma unroll
    for (int di = 0; di < D; ++di)
#pragma unroll
      for (int dj = 0; dj < D; ++dj) acc[di] += vals[vix<D, LAYOUT>(q, di * D + dj, nnzb)] * xj[dj];
  }
#pragma unroll
  for (int d = 0; d < D; ++d) acc[d] = group_sum<G>(acc[d]);
}

// 16-byte vectors: W = 16 / sizeof(T) consecutive entries of one value plane, and their columns.
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
  typedef float V __attribute__((ext_vector_type(4)));
  typedef int32_t I __attribute__((ext_vector_type(4)));
  static constexpr int W = 4;
};
template <>
struct Vec16<double> {
  typedef double V __attribute__((ext_vector_type(2)));
  typedef int32_t I __attribute__((ext_vector_type(2)));
  static constexpr int W = 2;
};

// Row product on a padded pattern (row_align = 4: every row starts at a multiple of 4 blocks and
// holds a multiple of 4; padding blocks are zero with the row as column).  G lanes per row; a lane
// takes W consecutive blocks per step, one 16-byte load per value plane and one for the columns.
// The summation order depends on the row alone (not on where the row sits in the arrays).
// active false: an empty row (the lanes still take part in the group's shuffles).
// The row's block range [s, e) as read from bptr (by the caller, e.g. ahead of a barrier).
template <typename T, int D, int G>
__device__ inline void bsr_row_vec_range(const int32_t* __restrict__ bcol, const T* __restrict__ vals,
                                         int64_t nnzb, const T* __restrict__ x, int32_t s, int32_t e,
                                         int lane, T (&acc)[D]) {
  using V = typename Vec16<T>::V;
  using I = typename Vec16<T>::I;
  constexpr int W = Vec16<T>::W;
#pragma unroll
  for (int d = 0; d < D; ++d) acc[d] = T(0);
  for (int32_t q = s + lane * W; q < e; q += G * W) {
    const I cols = *reinterpret_cast<const I*>(bcol + q);
    V a[D * D];
#pragma unroll
    for (int k = 0; k < D * D; ++k) a[k] = *reinterpret_cast<const V*>(vals + (int64_t)k * nnzb + q);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int64_t j = cols[w];
      T xj[D];
#pragma unroll
      for (int d = 0; d < D; ++d) xj[d] = x[j * D + d];
#pragma unroll
      for (int di = 0; di < D; ++di)
#pragma unroll
        for (int dj = 0; dj < D; ++dj) acc[di] += a[di * D + dj][w] * xj[dj];
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) acc[d] = group_sum<G>(acc[d]);
}

template <typename T, int D, int G>
__device__ inline void bsr_row_vec(const int32_t* __restrict__ bptr, const int32_t* __restrict__ bcol,
                                   const T* __restrict__ vals, int64_t nnzb, const T* __restrict__ x,
                                   int64_t i, int lane, T (&acc)[D], bool active = true) {
  const int32_t s = active ? bptr[i] : 0, e = active ? bptr[i + 1] : 0;
  bsr_row_vec_range<T, D, G>(bcol, vals, nnzb, x, s, e, lane, acc);
}

// Whether A is on a padded pattern the vector row product may walk.
inline bool row_aligned(const fe_bsr* A) { return A->layout == FE_LAYOUT_PLANES && A->row_align == 4; }

template <typename T, int D>
__device__ inline T pick(const T (&acc)[D], int lane) {
  T out = acc[0];
#pragma unroll
  for (int d = 1; d < D; ++d)
    if (lane == d) out = acc[d];
  return out;
}

template <int D>
constexpr int lanes_for() {
  return D == 3 ? 16 : 8;
}

inline int lanes_for_dof(int d) { return d == 3 ? 16 : 8; }

// Argument check shared by the sparse entry points.
inline int check_bsr(const fe_bsr* A, const char* who) {
  if (!A) return fe_set_error(FE_ERR_ARG, "%s: null matrix", who);
  if (A->dof < 1 || A->dof > 3) return fe_set_error(FE_ERR_ARG, "%s: dof must be 1..3", who);
  if (A->precision != 0 && A->precision != 1)
    return fe_set_error(FE_ERR_ARG, "%s: precision must be 0 (FP64) or 1 (FP32)", who);
  if (A->layout != FE_LAYOUT_BSR && A->layout != FE_LAYOUT_PLANES)
    return fe_set_error(FE_ERR_ARG, "%s: layout must be FE_LAYOUT_BSR or FE_LAYOUT_PLANES", who);
  if (A->n_brows < 0 || A->nnzb < 0) return fe_set_error(FE_ERR_ARG, "%s: negative sizes", who);
  if (A->row_align != 0) {
    if (A->row_align != 4 || A->layout != FE_LAYOUT_PLANES || A->nnzb % 4 != 0)
      return fe_set_error(FE_ERR_ARG, "%s: row_align must be 0, or 4 with FE_LAYOUT_PLANES and nnzb a "
                          "multiple of 4", who);
    if (((uintptr_t)A->bcol | (uintptr_t)A->vals) % 16 != 0)
      return fe_set_error(FE_ERR_ARG, "%s: row_align = 4 needs 16-byte aligned bcol and vals", who);
  }
  if (A->n_brows > 0 && (!A->bptr || !A->bcol || !A->vals))
    return fe_set_error(FE_ERR_ARG, "%s: null matrix array", who);
  return FE_OK;
}


}  // namespace fe_sparse
