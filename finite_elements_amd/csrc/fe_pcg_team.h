// The whole PCG solve of one system in one launch: a team of co-resident workgroups, one tile of rows per
// 256 threads, that meet at barriers in device memory instead of at kernel boundaries.
//
// What bounds it: latency.  A chip-resident system (up to kTeamMaxTiles tiles: 131,072 node rows with three
// DOF per node, 262,144 with one or two) spends its iteration on dependent launches -- 2.7 us each when
// empty, three per iteration (six with the coarse correction) -- and not on its few MB of matrix.  Here
// an iteration is two messages:
//   A  every workgroup stores its new u and reads the u of its columns that others own into LDS;
//   B  every workgroup stores its tiles' partial dots, reads everybody's, and forms the same sums, alpha
//      and beta itself.
// Everything that crosses workgroups is stored and loaded by agent-scope atomics, which pass the
// (per-XCD) L2s: agent-scope release and acquire fences write back and invalidate an L2 in every
// workgroup, 12 to 25 us per barrier of 256 workgroups.  A message word is 64 bits, half of it payload, half
// the iteration's number: a reader polls the data itself.  Against a flag stored after the data that saves
// two of three trips to memory of about 0.8 us (the wait for the data's stores, and the load after the
// flag).  The reliable updates (a few per solve) use flags.  The matrix, or where it is too wide its
// columns, stays in registers for the whole solve; vectors are in registers between updates.
// Per iteration, launched kernels and this: 40 x 10 plate FP64 (one workgroup) 11.2 -> 2.8 us, 13^3 cube
// FP64 (22 workgroups) 17 -> 6.6 us, 150^2 magnetostatics FP64 (90) 13.6 -> 5.4 us; two-level mixed 27^3 cube
// with shuffled nodes (172) 40 -> 14.3 us, 450^2 magnetostatics (199) 33 -> 12.7 us.
//
// Two-level preconditioner (CO): the node rows are numbered aggregate by aggregate (order), so that a
// workgroup's rows touch few aggregates.  The correction P A_c^-1 P^T r is carried by the recurrence of r:
// with z, zeta and y the corrections of r, s and w, s = w + beta s gives zeta = y + beta zeta and
// r -= alpha s gives z -= alpha zeta, so an iteration needs P^T w only.  Every tile sums its rows' share of
// P^T w by aggregate and hands it over with its partial dots; every workgroup adds all of them up and applies
// the rows of A_c^-1 that its own aggregates need.  The correction costs no further meeting (launched:
// three kernels per iteration).  The reliable updates form z, zeta and y anew, and in FP64, which has them at
// its convergence claims only, z is also formed anew each time |r| has fallen by 1,000, by one more meeting: the
// rounding of z -= alpha zeta does not shrink with r.  (Magnetostatics on 200 x 200 cells, ln mu of standard
// deviation 3, to 1e-10, mean of 12 right-hand sides: 2,032 iterations without, 1,661 with it, 1,636 by the
// launched kernels.)
// Shares, z, zeta and y are in the coarse space's orthonormal basis (P = Z T): the rigid-body moments and
// motions on the other side of T stay in FP64 inside a tile or an aggregate.  An aggregate of two nodes, or of
// nodes on a line, has T entries of 1e8, and a product such as T A_c^-1 T^T, a moment rounded to FP32 or a
// recurrence in the motions would lose the correction in them.
// All workgroups read all shares, a few KB that message words and agent-scope loads would fetch from
// memory once per workgroup (450^2 magnetostatics, 199 workgroups: 16 us per iteration).  So here the
// shares and dots are stored first, by agent-scope stores, then a flag, and read by plain loads, which
// the workgroups of an XCD share through its L2.  That is sound because a meeting's region of memory has not
// been read since the last invalidation: the regions are a ring of kTeamRing, and every wavefront
// invalidates (agent-scope acquire fence) before it reads the ring's first region; a workgroup's part of a
// region begins on a cache line of its own.
//
// The arithmetic -- tiles, row products, partial sums and their order, the scalars, reliable updates at
// chunk ends -- is that of the launched kernels (fe_pcg.hip), so a system solved here without a
// coarse correction has the bits of the same system solved as a segment of a batch.
//
// The launch of more than one workgroup is cooperative (all of them resident; a process' cooperative launches on
// a device take turns).  Every
// wait is bounded: a thread that has polled `spins` times notes it for its workgroup, whose waits, its own next
// ones among them, then end after 64 polls; the workgroup leaves at the end of the meeting and raises `abort`,
// which the others' waits look at as often, and the host finishes the solve with the launched kernels.
#pragma once

#include "fe_sparse.h"

namespace {

constexpr int kTeamMaxTiles = 1024;
constexpr int kTeamCopies = 8;  // of the partial dots: a workgroup reads copy blockIdx.x % 8
constexpr int kTeamMaxCoarse = 1536;  // coarse DOF: every workgroup holds all of P^T w in LDS
constexpr int kTeamRing = 64;   // regions of the shares' ring
constexpr double kTeamFresh = 1e-6;  // fall of r.r after which z is formed anew
constexpr int kTeamLds = 144 * 1024;  // dynamic LDS of a workgroup, of the CU's 160 KB

struct TeamArgs {
  int32_t n_rows, ntiles, pstride;  // node rows, tiles that hold them, stride of the partial arrays
  int64_t nnzb_it, nnzb;
  const int32_t *bptr_it, *bcol_it, *bptr, *bcol;
  const void* vit;
  const double* v64;
  const void* M;
  const double* b;
  double* x;
  void *r, *u, *w, *p, *s;
  double* r64;
  PcgState* st;
  double* partials;  // 2 x 5 arrays: meetings alternate between the halves
  uint64_t* flags;   // one per workgroup, zero before the launch
  int32_t* abort;    // zero before the launch
  int32_t spins;     // bound of a wait, in polls of about a microsecond
  uint64_t* ut;      // u as messages: sizeof(T) / 4 words per DOF
  uint64_t* pt;      // partial dots as messages: 2 halves x kTeamCopies x 6 words x pstride
  int32_t lds_remote;  // remote node rows whose u fits in LDS
  int32_t chunk;
  int64_t max_chunks;
  // two-level: node rows by aggregate (row i of the iteration matrix is node order[i]), the aggregates'
  // row ranges, their nodes' x^ and constraint bits, their T, A_c^-1 (iteration precision, leading
  // dimension lda) and the ring of kTeamRing regions of region bytes
  const int32_t *order, *agg_ptr, *node_agg;
  const void* xhat;
  const uint8_t* fixed_bits;
  const double* Tm;
  const void* Ainv;
  int64_t lda;
  int32_t n_agg;
  char* ring;
  int64_t region;
};

// A_c^-1 in FP32.
__global__ __launch_bounds__(256) void k_team_cast(int64_t n, const double* __restrict__ in, float* __restrict__ out) {
  const int64_t t = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (t < n) out[t] = (float)in[t];
}

// A region of the ring: workgroup b's three partial dots, then its parts, the first of them
// part q0; its place leaves whole cache lines to the workgroups before it.
inline __host__ __device__ int64_t team_part(int64_t b, int64_t q0, int NC, int elem) {
  return 128 * (2 * b + q0 * NC * elem / 128);
}
constexpr int kTeamDots = 32;  // bytes of the dots ahead of the parts

// Dynamic LDS of a workgroup: the parts beside u's, which take the rest.
struct TeamLds {
  int64_t bits, wl, xl, fb, ap, zs, total;  // byte offsets from the end of rlist, and their sum
};
inline __host__ __device__ TeamLds team_lds(int64_t n_rows, int64_t wg_rows, int64_t n_agg, int D, int NC, int elem) {
  TeamLds l{};
  auto take = [&](int64_t& at, int64_t bytes) {
    at = l.total;
    l.total += (bytes + 15) / 16 * 16;
  };
  take(l.bits, (n_rows + 31) / 32 * 6);
  if (n_agg > 0) {
    take(l.wl, wg_rows * D * elem);
    take(l.xl, D == 1 ? 0 : wg_rows * 3 * elem);
    take(l.fb, wg_rows);
    take(l.ap, (n_agg + 1) * 4);
    take(l.zs, n_agg * NC * 8);
  }
  return l;
}

template <typename V>
__device__ inline V ld_team(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ inline void st_team(V* p, V v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Keeps an accumulator's entries in registers (a lane's choice among them would otherwise become an index).
template <typename T, int D>
__device__ inline void in_registers(T (&v)[D]) {
#pragma unroll
  for (int d = 0; d < D; ++d) asm volatile("" : "+v"(v[d]));
}

// v, in a form the compiler cannot move: addresses formed from it are formed where they are used instead of
// being kept in registers (two each, per array and pass) over the whole solve.
__device__ inline int32_t team_here(int32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Raise abort: 1 a wait reached its bound, 2 a workgroup's columns do not fit in its LDS (which stays 2).
__device__ inline void team_give_up(int32_t* abort, int32_t why) {
  __hip_atomic_fetch_max(abort, why, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Poll until `ready()`; false, noted in *fail, when the bound is reached or this or another workgroup has given
// up.  (Raising abort here as well costs registers at every poll: the four-tile kernels spilled twice as many.)
template <typename F>
__device__ inline bool team_poll(const int32_t* abort, int32_t spins, int* fail, F ready) {
  for (int32_t n = 0; n < spins; ++n) {
    if (ready()) return true;
    if ((n & 63) == 63 && (ld_team(abort) != 0 || *(volatile int*)fail)) break;
  }
  *(volatile int*)fail = 1;
  return false;
}

// A message: a value's 32-bit pieces, each in a word with the iteration's number.
template <typename V>
constexpr int team_words() { return (int)sizeof(V) / 4; }

__device__ inline void team_put(uint64_t* m, uint32_t tag, float v) {
  st_team(m, ((uint64_t)tag << 32) | __float_as_uint(v));
}
__device__ inline void team_put(uint64_t* m, uint32_t tag, double v, int stride = 1) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  st_team(m, ((uint64_t)tag << 32) | (uint32_t)b);
  st_team(m + stride, ((uint64_t)tag << 32) | (uint32_t)(b >> 32));
}
__device__ inline bool team_got(const uint64_t* w, int n, uint32_t tag) {
  bool ok = true;
#pragma unroll
  for (int k = 0; k < n; ++k) ok = ok && (uint32_t)(w[k] >> 32) == tag;
  return ok;
}
__device__ inline float team_value(const uint64_t (&w)[1]) { return __uint_as_float((uint32_t)w[0]); }
__device__ inline double team_value(const uint64_t (&w)[2]) {
  return __longlong_as_double((long long)((w[1] << 32) | (uint32_t)w[0]));
}

// Whether a thread's share of the iteration matrix (the first vector step of every row) stays in its
// registers, by what the workgroup size leaves a thread.
template <typename T, int D, int S>
constexpr bool team_resident() {
  constexpr int W = Vec16<T>::W, GV = lanes_for<D>() / W;
  constexpr int passes = tile_rows<lanes_for<D>()>() / (kBlock / GV);
  constexpr int regs = passes * W * (D * D * (int)sizeof(T) / 4 + 1);
  return regs <= (S == 1 ? 168 : S == 2 ? 80 : 40);
}

template <typename T, int D, int PC, int S, bool CO>
__global__ __launch_bounds__(kBlock* S) void k_pcg_team(TeamArgs a) {
  using V = typename Vec16<T>::V;
  using I = typename Vec16<T>::I;
  constexpr int W = Vec16<T>::W;
  constexpr int G = lanes_for<D>(), GV = G / W;   // lanes per row: own and padded pattern
  constexpr int R = tile_rows<G>();               // rows per tile
  constexpr int kRows = kBlock / GV;              // rows per pass of the iteration's row product
  constexpr int kPasses = R / kRows;
  constexpr int NM = PC == FE_PC_JACOBI ? 1 : D;
  constexpr int NC = D == 1 ? 1 : D == 2 ? 3 : 6;  // rigid-body modes of an aggregate
  constexpr int NT = kBlock * S;
  constexpr int TW = team_words<T>();
  constexpr bool kRes = team_resident<T, D, S>();
  constexpr int kWaves = kBlock / 64;
  static_assert(kPasses * kRows == R, "tile = whole passes");

  __shared__ PcgState st;  // written by thread 0: every workgroup's sums, and so its scalars, are the same
  __shared__ double s_red[S][5][kWaves];
  __shared__ double s_sum[5][kWaves];
  __shared__ int s_fail, s_lo, s_hi;
  constexpr bool kFresh = CO && sizeof(T) == 8;
  __shared__ double s_top;  // largest r.r since z was last formed from r (thread 0)
  __shared__ int s_fresh;   // form it in this iteration
  __shared__ int s_scan[NT];
  __shared__ int s_q0[CO ? 256 : 1];
  // u by local row: this workgroup's S R rows, then the rows of others that its blocks touch (rlist,
  // ascending); a bit per row of the system for the latter, and the number of bits before each word
  extern __shared__ __align__(16) char s_dyn[];
  T* ul = (T*)s_dyn;
  int32_t* rlist = (int32_t*)(s_dyn + (size_t)(S * R + a.lds_remote) * D * sizeof(T));
  char* s_rest = (char*)(rlist + a.lds_remote);
  const TeamLds at_lds = team_lds(a.n_rows, S * R, CO ? a.n_agg : 0, D, NC, (int)sizeof(T));
  uint32_t* bits = (uint32_t*)(s_rest + at_lds.bits);
  const int nwords = (a.n_rows + 31) / 32;
  uint16_t* rank = (uint16_t*)(bits + nwords);
  // two-level: a vector and the nodes' x^ and constraint bits by own row, the aggregates' row ranges and the
  // coarse vectors
  T* wl_ = (T*)(s_rest + at_lds.wl);
  T* xl = (T*)(s_rest + at_lds.xl);
  uint8_t* fb = (uint8_t*)(s_rest + at_lds.fb);
  int32_t* aggp = (int32_t*)(s_rest + at_lds.ap);
  double* cm = (double*)(s_rest + at_lds.zs);

  const int sub = threadIdx.x / kBlock, tid = threadIdx.x % kBlock;
  const int wl = threadIdx.x & 63, wid = tid >> 6;
  const int tile = blockIdx.x * S + sub;
  const bool alone = gridDim.x == 1;
  const int32_t row0 = (int32_t)min((int64_t)tile * R, (int64_t)a.n_rows);
  const int32_t row1 = (int32_t)min((int64_t)row0 + R, (int64_t)a.n_rows);
  const int32_t wr0 = (int32_t)min((int64_t)blockIdx.x * S * R, (int64_t)a.n_rows);
  const int32_t wr1 = (int32_t)min((int64_t)wr0 + S * R, (int64_t)a.n_rows);
  const int lane = tid % GV, lane_it = tid % G;
  const T* __restrict__ M = (const T*)a.M;
  const T* __restrict__ vit = (const T*)a.vit;
  T* u = (T*)a.u;
  T* p = (T*)a.p;
  T* r = (T*)a.r;
  T* w = (T*)a.w;
  T* s = (T*)a.s;

  // ---- plan: which rows of others this workgroup reads, and its blocks' columns as local rows -----------
  if (threadIdx.x == 0) {
    st = *a.st;
    s_fail = 0;
    s_lo = (int)gridDim.x;
    s_hi = -1;
  }
  for (int k = threadIdx.x; k < nwords; k += NT) bits[k] = 0;
  __syncthreads();
  int32_t rs[kPasses], re[kPasses];
  int lo = (int)gridDim.x, hi = -1;
#pragma unroll
  for (int ps = 0; ps < kPasses; ++ps) {
    const int32_t i = row0 + ps * kRows + tid / GV;
    const bool ok = i < row1;
    rs[ps] = ok ? a.bptr_it[i] : 0;
    re[ps] = ok ? a.bptr_it[i + 1] : 0;
    for (int32_t q = rs[ps] + lane * W; q < re[ps]; q += GV * W) {
      const I cols = *reinterpret_cast<const I*>(a.bcol_it + q);
#pragma unroll
      for (int k = 0; k < W; ++k) {
        lo = min(lo, cols[k] / (R * S));
        hi = max(hi, cols[k] / (R * S));
        if (cols[k] < wr0 || cols[k] >= wr1) atomicOr(&bits[cols[k] >> 5], 1u << (cols[k] & 31));
      }
    }
  }
  atomicMin(&s_lo, lo);
  atomicMax(&s_hi, hi);
  __syncthreads();
  lo = s_lo;
  hi = s_hi;
  const int per = (nwords + NT - 1) / NT, w0 = min((int)threadIdx.x * per, nwords), w1 = min(w0 + per, nwords);
  int count = 0;
  for (int k = w0; k < w1; ++k) count += __popc(bits[k]);
  s_scan[threadIdx.x] = count;
  __syncthreads();
  for (int off = 1; off < NT; off <<= 1) {
    const int add = (int)threadIdx.x >= off ? s_scan[threadIdx.x - off] : 0;
    __syncthreads();
    s_scan[threadIdx.x] += add;
    __syncthreads();
  }
  const int nr = s_scan[NT - 1];  // remote rows
  // two-level: behind the remote rows' u, the coarse vectors and T of the workgroup's aggregates
  int g0 = 0, ng = 0;
  if constexpr (CO) {
    g0 = a.node_agg[a.order[wr0]];
    ng = (wr1 > wr0 ? a.node_agg[a.order[wr1 - 1]] : g0) - g0 + 1;
  }
  const int co_rows = ((4 + NC) * ng * NC * 8 + 16 + D * (int)sizeof(T) - 1) / (D * (int)sizeof(T));  // in rows of u
  const bool fits = nr + (CO ? co_rows : 0) <= a.lds_remote;
  int at = s_scan[threadIdx.x] - count;
  for (int k = w0; k < w1; ++k) {
    rank[k] = (uint16_t)at;
    for (uint32_t m = bits[k]; m; m &= m - 1, ++at)
      if (fits) rlist[at] = k * 32 + __ffs(m) - 1;
  }
  __syncthreads();
  auto local_row = [&](int32_t col) -> int32_t {
    if (col >= wr0 && col < wr1) return col - wr0;
    return S * R + (int32_t)rank[col >> 5] + (int32_t)__popc(bits[col >> 5] & ((1u << (col & 31)) - 1u));
  };
  // this thread's share of the first vector step of its rows, and its DOF's preconditioner row
  V av[kRes ? kPasses : 1][D * D];
  I cv[kPasses];
  T mk[kPasses][NM];
#pragma unroll
  for (int ps = 0; ps < kPasses; ++ps) {
    const int32_t i = row0 + ps * kRows + tid / GV;
#pragma unroll
    for (int j = 0; j < NM; ++j) mk[ps][j] = T(0);
    if (i < row1 && lane < D) {
      const int64_t node = CO ? a.order[i] : i;
      const T* m = PC == FE_PC_JACOBI ? M + node * D + lane : M + node * D * D + lane * D;
#pragma unroll
      for (int j = 0; j < NM; ++j) mk[ps][j] = m[j];
    }
    const int32_t q = rs[ps] + lane * W;
    if (q < re[ps]) {
      const I cols = *reinterpret_cast<const I*>(a.bcol_it + q);
#pragma unroll
      for (int k = 0; k < W; ++k) cv[ps][k] = local_row(cols[k]);
      if constexpr (kRes)
#pragma unroll
        for (int k = 0; k < D * D; ++k) av[ps][k] = *reinterpret_cast<const V*>(vit + (int64_t)k * a.nnzb_it + q);
    }
  }

  uint64_t epoch = 0;
  int half = 0;  // of the partial arrays
  // The stores of this workgroup's threads are complete before its flag is.
  auto arrive = [&]() {
    ++epoch;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) st_team(a.flags + blockIdx.x, epoch);
  };
  // A: after the stores of u (or x, or p), wait for the owners of this workgroup's columns.
  auto meet_neighbours = [&]() {
    arrive();
    for (int g = lo + (int)threadIdx.x; g <= hi; g += NT)
      team_poll(a.abort, a.spins, &s_fail, [&] { return ld_team(a.flags + g) >= epoch; });
    __syncthreads();
    return s_fail == 0;
  };
  // B: the tile's NV partial sums (v of every thread) stored, then v the sums over all tiles, in every
  // thread.  The order of both sums is that of block_sum and seg_sum.
  auto meet_all = [&](auto& v) {
    constexpr int NV = sizeof(v) / sizeof(double);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      v[k] = wave_sum(v[k]);
      if (wl == 0) s_red[sub][k][wid] = v[k];
    }
    __syncthreads();
    double* part = a.partials + (int64_t)half * 5 * a.pstride;
    if (tid < NV && tile < a.ntiles) {
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) t += s_red[sub][tid][q];
      st_team(part + (int64_t)tid * a.pstride + tile, t);
    }
    arrive();
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = 0.0;
    if (sub == 0) {
      for (int t = tid; t < a.ntiles; t += kBlock)
        team_poll(a.abort, a.spins, &s_fail, [&] { return ld_team(a.flags + t / S) >= epoch; });
      // at most S kBlock tiles: one per workgroup of S subgroups, one workgroup per CU
      double e[S][NV];
#pragma unroll
      for (int j = 0; j < S; ++j)
#pragma unroll
        for (int k = 0; k < NV; ++k)
          e[j][k] = tid + j * kBlock < a.ntiles ? ld_team(part + (int64_t)k * a.pstride + tid + j * kBlock) : 0.0;
#pragma unroll
      for (int j = 0; j < S; ++j)
        if (tid + j * kBlock < a.ntiles)
#pragma unroll
          for (int k = 0; k < NV; ++k) v[k] += e[j][k];
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        v[k] = wave_sum(v[k]);
        if (wl == 0) s_sum[k][wid] = v[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) t += s_sum[k][q];
      v[k] = t;
    }
    half ^= 1;
    return s_fail == 0;
  };

  uint32_t tag = 0;  // of this iteration's messages
  // A of an iteration: uk to this workgroup's LDS and to the others, theirs to LDS.
  auto exchange_u = [&](const T* uk) {
    ++tag;
#pragma unroll
    for (int ps = 0; ps < kPasses; ++ps) {
      const int32_t i = team_here(row0 + tid / GV) + ps * kRows;
      if (lane >= D || i >= row1) continue;
      ul[(i - wr0) * D + lane] = uk[ps];
      if (!alone) team_put(a.ut + ((int64_t)i * D + lane) * TW, tag, uk[ps]);
    }
    constexpr int B = (S == 4 ? 4 : 8) / TW;  // messages of a thread in flight together
    for (int e0 = threadIdx.x; e0 < nr * D; e0 += NT * B) {
      uint64_t m[B][TW];
      const uint64_t* from[B];
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int e = min(e0 + j * NT, nr * D - 1);
        from[j] = a.ut + ((int64_t)rlist[e / D] * D + e % D) * TW;
#pragma unroll
        for (int h = 0; h < TW; ++h) m[j][h] = ld_team(from[j] + h);
      }
#pragma unroll
      for (int j = 0; j < B; ++j) {
        if (e0 + j * NT >= nr * D) break;
        if (!team_got(m[j], TW, tag)) team_poll(a.abort, a.spins, &s_fail, [&] {
#pragma unroll
          for (int h = 0; h < TW; ++h) m[j][h] = ld_team(from[j] + h);
          return team_got(m[j], TW, tag);
        });
        ul[S * R * D + e0 + j * NT] = team_value(m[j]);
      }
    }
    __syncthreads();
    return s_fail == 0;
  };
  // B of an iteration: meet_all's sums of three values, by messages.
  auto exchange_dots = [&](double (&v)[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      v[k] = wave_sum(v[k]);
      if (wl == 0) s_red[sub][k][wid] = v[k];
    }
    __syncthreads();
    auto tile_sum = [&](int sb, int k) {
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) t += s_red[sb][k][q];
      return t;
    };
    if (alone) {
      // the butterfly over one or two tiles and zeros, written out (four are in one of many workgroups)
#pragma unroll
      for (int k = 0; k < 3; ++k) v[k] = S == 1 ? tile_sum(0, k) : tile_sum(0, k) + tile_sum(S - 1, k);
      return true;
    }
    uint64_t* box = a.pt + (int64_t)(tag & 1) * (6 * kTeamCopies) * a.pstride;
    if (tid < 3 * kTeamCopies && tile < a.ntiles)
      team_put(box + (int64_t)2 * tid * a.pstride + tile, tag, tile_sum(sub, tid % 3), a.pstride);
    if (sub == 0) {
      const uint64_t* in = box + (int64_t)(blockIdx.x % kTeamCopies) * 6 * a.pstride;
      uint64_t m[S][3][2];
      auto load = [&](int j) {
        const int t = min(tid + j * kBlock, a.ntiles - 1);
#pragma unroll
        for (int k = 0; k < 6; ++k) m[j][k / 2][k % 2] = ld_team(in + (int64_t)k * a.pstride + t);
      };
      auto got = [&](int j) { return team_got(m[j][0], 2, tag) && team_got(m[j][1], 2, tag) && team_got(m[j][2], 2, tag); };
#pragma unroll
      for (int j = 0; j < S; ++j) load(j);
#pragma unroll
      for (int k = 0; k < 3; ++k) v[k] = 0.0;
#pragma unroll
      for (int j = 0; j < S; ++j) {
        if (tid + j * kBlock >= a.ntiles) break;
        if (!got(j)) team_poll(a.abort, a.spins, &s_fail, [&] { load(j); return got(j); });
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] += team_value(m[j][k]);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        v[k] = wave_sum(v[k]);
        if (wl == 0) s_sum[k][wid] = v[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) t += s_sum[k][q];
      v[k] = t;
    }
    return s_fail == 0;
  };

  // the owned DOFs' vectors (lane < D): in registers while the segment iterates
  T pk[kPasses], sk[kPasses], rk[kPasses], wk[kPasses], uk[kPasses];
  double xk[kPasses];
  const int32_t my_row = row0 + tid / GV;
  auto own = [&](int ps, int64_t& k) {
    const int32_t i = team_here(my_row) + ps * kRows;
    k = (int64_t)i * D + lane;
    return lane < D && i < row1;
  };
  // the DOF's place in the caller's vectors (x, b)
  auto caller = [&](int ps, int64_t k) -> int64_t {
    if constexpr (!CO) return k;
    return (int64_t)a.order[team_here(my_row) + ps * kRows] * D + lane;
  };
#pragma unroll
  for (int ps = 0; ps < kPasses; ++ps) {
    int64_t k;
    pk[ps] = sk[ps] = rk[ps] = wk[ps] = uk[ps] = T(0);
    xk[ps] = 0.0;
    if (own(ps, k)) {
      xk[ps] = a.x[caller(ps, k)];
      // words of an earlier solve could carry this one's numbers: cleared ahead of the first meeting
#pragma unroll
      for (int h = 0; h < TW; ++h) st_team(a.ut + k * TW + h, (uint64_t)0);
    }
  }
  if (tid < 12 * kTeamCopies && tile < a.ntiles) st_team(a.pt + (int64_t)tid * a.pstride + tile, (uint64_t)0);
  // u = M r of the owned DOFs; the node's residuals come from its group's lanes
  auto precond = [&]() {
#pragma unroll
    for (int ps = 0; ps < kPasses; ++ps) {
      if constexpr (PC == FE_PC_JACOBI) {
        uk[ps] = mk[ps][0] * rk[ps];
      } else {
        T t = T(0);
        t += mk[ps][0] * group_lane<GV, 0>(rk[ps]);
        if constexpr (D > 1) t += mk[ps][(D > 1 ? 1 : 0)] * group_lane<GV, 1>(rk[ps]);
        if constexpr (D > 2) t += mk[ps][(D > 2 ? 2 : 0)] * group_lane<GV, (D > 2 ? 2 : 0)>(rk[ps]);
        uk[ps] = t;
      }
    }
  };

  // ---- coarse correction (CO) -----------------------------------------------------------------------
  const int n_c = CO ? a.n_agg * NC : 0;
  double* zc = (double*)(s_dyn + (((size_t)(S * R + nr) * D * sizeof(T) + 15) & ~(size_t)15));
  double *ze = zc + ng * NC, *yc = ze + ng * NC, *ym = yc + ng * NC, *tl = ym + ng * NC;
  int tg0 = 0, tg1 = -1;
  if constexpr (CO) {
    // the tile's parts: its aggregates, from that of the row before it (an empty part where the tile starts
    // one), so that the parts of all tiles are numbered tile + aggregate without a gap
    if (tile < a.ntiles) {
      tg0 = row0 > 0 ? a.node_agg[a.order[row0 - 1]] : 0;
      tg1 = a.node_agg[a.order[row1 - 1]];
    }
    for (int32_t i = wr0 + (int)threadIdx.x; i < wr1; i += NT) {
      const int64_t node = a.order[i];
      fb[i - wr0] = a.fixed_bits[node];
      if constexpr (D > 1)
#pragma unroll
        for (int c = 0; c < 3; ++c) xl[(i - wr0) * 3 + c] = ((const T*)a.xhat)[node * 3 + c];
    }
    if (fits)
      for (int e = threadIdx.x; e < ng * NC * NC; e += NT) tl[e] = a.Tm[(int64_t)g0 * NC * NC + e];
  }
  int32_t la[kPasses];  // first of the node's aggregate's entries in ym, or -1 where the DOF is constrained
#pragma unroll
  for (int ps = 0; ps < kPasses; ++ps) {
    la[ps] = -1;
    if constexpr (CO) {
      const int32_t i = row0 + ps * kRows + tid / GV;
      if (lane < D && i < row1) {
        const int32_t node = a.order[i];
        if (!((a.fixed_bits[node] >> lane) & 1)) la[ps] = (a.node_agg[node] - g0) * NC;
      }
    }
  }
  const int nwg = (int)gridDim.x;
  if constexpr (CO)
    for (int g = threadIdx.x; g < nwg; g += NT) {
      const int32_t row = g * S * R;
      s_q0[g] = g * S + (row > 0 ? a.node_agg[a.order[row - 1]] : 0);
    }
  if constexpr (CO)
    for (int g = threadIdx.x; g <= a.n_agg; g += NT) aggp[g] = a.agg_ptr[g];
  constexpr int kParts = 2;
  int turn = 0;  // region of the ring
  // the rows of A_c^-1 that this workgroup applies, in LDS behind the remote rows where they fit
  const T* Arows = (const T*)a.Ainv + (int64_t)g0 * NC * a.lda;
  int64_t lda = a.lda;
  if constexpr (CO) {
    if (fits && (int64_t)ng * NC * n_c <= (int64_t)(a.lds_remote - nr - co_rows) * D) {
      T* Al = (T*)(tl + ng * NC * NC);
      for (int q = (int)threadIdx.x / 64; q < ng * NC; q += NT / 64)
        for (int c = wl; c < n_c; c += 64) Al[q * n_c + c] = Arows[q * lda + c];
      Arows = Al;
      lda = n_c;
    }
  }
  auto coarse_rows = [&](const T* v) {
#pragma unroll
    for (int ps = 0; ps < kPasses; ++ps) {
      const int32_t i = team_here(my_row) + ps * kRows;
      if (lane < D && i < row1) wl_[(i - wr0) * D + lane] = v[ps];
    }
  };
  // A meeting of all for P^T of the rows in wl_ and, if v3, the dots' wavefront sums in s_red (both
  // behind a barrier): P^T w in cm, the dots' sums over the workgroups' wavefronts in s_sum.
  auto coarse_meet = [&](bool dots) {
    char* region = a.ring + turn * a.region;
    if (++turn == kTeamRing) turn = 0;
    const int q0 = s_q0[blockIdx.x];
    char* mine = region + team_part(blockIdx.x, q0, NC, (int)sizeof(T));
    auto put = [&](auto* to, auto v) {
      if (alone)
        *to = v;
      else
        st_team(to, v);
    };
    for (int g = tg0 + wid; g <= tg1; g += kWaves) {  // one part per wavefront at a time
      const int32_t p0 = max(row0, aggp[g]), p1 = min(row1, aggp[g + 1]);
      double m[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) m[c] = 0.0;
      for (int32_t i = p0 + wl; i < p1; i += 64) {
        const int l = i - wr0, bits_ = fb[l];
        double rv[D];
#pragma unroll
        for (int e = 0; e < D; ++e) rv[e] = ((bits_ >> e) & 1) ? 0.0 : (double)wl_[l * D + e];
        if constexpr (D == 3) {
          const double x = xl[l * 3], y = xl[l * 3 + 1], z = xl[l * 3 + 2];
          m[0] += rv[0];
          m[1] += rv[1];
          m[2] += rv[2];
          m[3] += y * rv[2] - z * rv[1];
          m[4] += z * rv[0] - x * rv[2];
          m[5] += x * rv[1] - y * rv[0];
        } else if constexpr (D == 2) {
          m[0] += rv[0];
          m[1] += rv[1];
          m[2] += (double)xl[l * 3] * rv[1] - (double)xl[l * 3 + 1] * rv[0];
        } else {
          m[0] += rv[0];
        }
      }
      // T^T of the moments (an empty part may be of the aggregate before the workgroup's first)
      double mine_c = 0.0;
      const double* tg = tl + (max(g, g0) - g0) * NC * NC + min(wl, NC - 1);
#pragma unroll
      for (int c = 0; c < NC; ++c) mine_c += tg[c * NC] * wave_sum(m[c]);
      if (wl < NC) put((T*)(mine + kTeamDots) + (tile + g - q0) * NC + wl, (T)mine_c);
    }
    if (dots && threadIdx.x < 3) {
      double t = 0.0;
#pragma unroll
      for (int sb = 0; sb < S; ++sb)
#pragma unroll
        for (int q = 0; q < kWaves; ++q) t += s_red[sb][threadIdx.x][q];
      put((double*)mine + threadIdx.x, t);
    }
    if (alone) {
      __syncthreads();
    } else {
      arrive();
      for (int g = threadIdx.x; g < nwg; g += NT)
        team_poll(a.abort, a.spins, &s_fail, [&] { return ld_team(a.flags + g) >= epoch; });
      __syncthreads();
      if (turn == 1) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // the ring's first region, also the first time
    }
    if (dots && sub == 0) {
      double e[3];
#pragma unroll
      for (int k = 0; k < 3; ++k)
        e[k] = tid < nwg ? ((const double*)(region + team_part(tid, s_q0[tid], NC, (int)sizeof(T))))[k] : 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        e[k] = wave_sum(e[k]);
        if (wl == 0) s_sum[k][wid] = e[k];
      }
    }
    // the parts t + g of the tiles t that touch aggregate g
    for (int e = threadIdx.x; e < n_c; e += NT) {
      const int g = e / NC, c = e % NC;
      const int t0 = aggp[g] / R, t1 = min(aggp[g + 1] / R, a.ntiles - 1);
      double v = 0.0;
      for (int t = t0; t <= t1; t += kParts) {
        T part[kParts];
#pragma unroll
        for (int j = 0; j < kParts; ++j) {
          const int tj = min(t + j, t1), q = s_q0[tj / S];
          part[j] = ((const T*)(region + team_part(tj / S, q, NC, (int)sizeof(T)) + kTeamDots))[(tj + g - q) * NC + c];
        }
#pragma unroll
        for (int j = 0; j < kParts; ++j) v += t + j <= t1 ? (double)part[j] : 0.0;
      }
      cm[e] = v;
    }
    __syncthreads();
    return s_fail == 0;
  };
  // (behind a barrier) out = A_c^-1 cm for the workgroup's aggregates, one wavefront per row
  auto coarse_apply_rows = [&](double* out) {
    for (int q = (int)threadIdx.x / 64; q < ng * NC; q += NT / 64) {
      const T* row = Arows + q * lda;
      double v = 0.0;
#pragma unroll 8
      for (int c = wl; c < n_c; c += 64) v += (double)row[c] * cm[c];
      v = wave_sum(v);
      if (wl == 0) out[q] = v;
    }
  };
  // out = A_c^-1 P^T v, a meeting of its own (reliable updates)
  auto coarse_round = [&](const T* v, double* out) {
    coarse_rows(v);
    __syncthreads();
    if (!coarse_meet(false)) return false;
    coarse_apply_rows(out);
    __syncthreads();
    return s_fail == 0;
  };
  // The rigid-body motions ym = T z of the workgroup's aggregates, z = zc after step(entry) has brought it up to
  // date; an aggregate's entries are neighbouring lanes'.
  auto coarse_motions = [&](auto step) {
    constexpr int L = NC == 6 ? 8 : NC == 3 ? 4 : 1;
    for (int e = threadIdx.x; e < ng * L; e += NT) {
      const int q = e / L * NC + min(e % L, NC - 1);
      const bool on = e % L < NC;
      const double z = on ? step(q) : 0.0;
      const double* t = tl + q * NC;
      double y = 0.0;
#pragma unroll
      for (int k = 0; k < NC; ++k) y += t[k] * (L == 1 ? z : __shfl(z, k, L));
      if (on) ym[q] = y;
    }
    __syncthreads();
  };
  // u += the rigid-body motion of the node's aggregate, on free DOFs
  auto coarse_add = [&]() {
#pragma unroll
    for (int ps = 0; ps < kPasses; ++ps) {
      if (la[ps] < 0) continue;
      const int l = team_here(my_row) + ps * kRows - wr0;
      const double* y = ym + la[ps];
      double du = y[lane];
      if constexpr (D == 3) {
        // lane 0: z w_y - y w_z, lane 1: x w_z - z w_x, lane 2: y w_x - x w_y
        const int n1 = lane == 2 ? 0 : lane + 1, n2 = lane == 0 ? 2 : lane - 1;
        du += (double)xl[l * 3 + n2] * y[3 + n1] - (double)xl[l * 3 + n1] * y[3 + n2];
      } else if constexpr (D == 2) {
        du += lane == 0 ? -(double)xl[l * 3 + 1] * y[2] : (double)xl[l * 3] * y[2];
      }
      uk[ps] += (T)du;
    }
  };

  int64_t chunks = 0;
  bool alive = fits;
  while (alive) {
    // ---- reliable update: the first one forms the starting residual ---------------------------------
    if (st.need_ru && !st.done) {
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        int64_t k;
        if (own(ps, k)) st_team(a.x + caller(ps, k), xk[ps]);
      }
      if (!meet_neighbours()) { alive = false; break; }
      double v1[1] = {0.0};
#pragma unroll 1
      for (int32_t i = row0 + team_here(tid) / G; i < row1; i += kBlock / G) {
        double acc[D];
#pragma unroll
        for (int d = 0; d < D; ++d) acc[d] = 0.0;
        const int64_t node = CO ? a.order[i] : i;
        for (int32_t q = a.bptr[node] + lane_it; q < a.bptr[node + 1]; q += G) {
          const int64_t j = a.bcol[q];
          double xj[D];
#pragma unroll
          for (int d = 0; d < D; ++d) xj[d] = ld_team(a.x + j * D + d);
#pragma unroll
          for (int di = 0; di < D; ++di)
#pragma unroll
            for (int dj = 0; dj < D; ++dj)
              acc[di] += a.v64[vix<D, FE_LAYOUT_PLANES>(q, di * D + dj, a.nnzb)] * xj[dj];
        }
#pragma unroll
        for (int d = 0; d < D; ++d) acc[d] = group_sum<G>(acc[d]);
        in_registers(acc);
        if (lane_it < D) {
          const int64_t k = (int64_t)i * D + lane_it;
          const double ri = a.b[node * D + lane_it] - pick<double, D>(acc, lane_it);
          a.r64[k] = ri;
          v1[0] += ri * ri;
        }
      }
      if (!meet_all(v1)) { alive = false; break; }
      if (threadIdx.x == 0) ru_decide(&st, v1[0]);
      __syncthreads();
      if (st.done) break;
      const bool first = st.first != 0;
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        int64_t k;
        if (!own(ps, k)) continue;
        rk[ps] = (T)a.r64[k];
        if (first) pk[ps] = sk[ps] = T(0);
      }
      if constexpr (CO) {
        if (!coarse_round(rk, zc)) { alive = false; break; }
        coarse_motions([&](int q) { return zc[q]; });
      }
      precond();
      if constexpr (CO) coarse_add();
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        int64_t k;
        if (!own(ps, k)) continue;
        r[k] = rk[ps];
        st_team(u + k, uk[ps]);
        st_team(p + k, pk[ps]);
      }
      if (!meet_neighbours()) { alive = false; break; }
      double v5[5] = {0, 0, 0, 0, 0};
#pragma unroll 1
      for (int32_t i = row0 + team_here(tid) / G; i < row1; i += kBlock / G) {
        T au[D], ap[D];
#pragma unroll
        for (int d = 0; d < D; ++d) au[d] = ap[d] = T(0);
        for (int32_t q = a.bptr_it[i] + lane_it; q < a.bptr_it[i + 1]; q += G) {
          const int64_t j = a.bcol_it[q];
          T uj[D], pj[D];
#pragma unroll
          for (int d = 0; d < D; ++d) {
            uj[d] = ld_team(u + j * D + d);
            pj[d] = ld_team(p + j * D + d);
          }
#pragma unroll
          for (int di = 0; di < D; ++di)
#pragma unroll
            for (int dj = 0; dj < D; ++dj) {
              const T m = vit[vix<D, FE_LAYOUT_PLANES>(q, di * D + dj, a.nnzb_it)];
              au[di] += m * uj[dj];
              ap[di] += m * pj[dj];
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
          au[d] = group_sum<G>(au[d]);
          ap[d] = group_sum<G>(ap[d]);
        }
        in_registers(au);
        in_registers(ap);
        if (lane_it < D) {
          const int64_t k = (int64_t)i * D + lane_it;
          const T wi = pick<T, D>(au, lane_it), si = pick<T, D>(ap, lane_it);
          w[k] = wi;
          s[k] = si;
          const double ui = ld_team(u + k), pi = ld_team(p + k), ri = r[k];
          v5[0] += ri * ui;
          v5[1] += ui * (double)wi;
          v5[2] += ui * (double)si;
          v5[3] += pi * (double)si;
          v5[4] += ri * ri;
        }
      }
      if (!meet_all(v5)) { alive = false; break; }
      if (threadIdx.x == 0) ru_finish(&st, v5);
      __syncthreads();
      if (st.done) break;
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        int64_t k;
        if (!own(ps, k)) continue;
        wk[ps] = w[k];
        sk[ps] = s[k];
      }
      if (kFresh && threadIdx.x == 0) {
        s_top = st.rr;
        s_fresh = 0;
      }
      if constexpr (CO) {
        if (!coarse_round(wk, yc) || !coarse_round(sk, ze)) { alive = false; break; }
      }
    }
    // ---- a chunk of iterations ----------------------------------------------------------------------
    if (st.done || ++chunks > a.max_chunks) break;
    for (int it = 0; it < a.chunk; ++it) {
      const double alpha = st.alpha;
      const T alpha_t = (T)alpha, beta = (T)st.beta;
      if constexpr (CO) {
        coarse_motions([&](int q) {
          ze[q] = yc[q] + st.beta * ze[q];
          return zc[q] -= alpha * ze[q];
        });
      }
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        pk[ps] = uk[ps] + beta * pk[ps];
        sk[ps] = wk[ps] + beta * sk[ps];
        xk[ps] = xk[ps] + alpha * (double)pk[ps];
        rk[ps] = rk[ps] - alpha_t * sk[ps];
      }
      if constexpr (kFresh) {
        if (s_fresh) {  // uniform over all workgroups, as the scalars are
          if (!coarse_round(rk, zc)) { alive = false; break; }
          coarse_motions([&](int q) { return zc[q]; });
        }
      }
      precond();
      if constexpr (CO) coarse_add();
      if (!exchange_u(uk)) { alive = false; break; }
      double v3[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int ps = 0; ps < kPasses; ++ps) {
        T acc[D];
#pragma unroll
        for (int d = 0; d < D; ++d) acc[d] = T(0);
        auto step = [&](const I& rows, const V (&m)[D * D]) {
#pragma unroll
          for (int k = 0; k < W; ++k) {
            T xj[D];
#pragma unroll
            for (int d = 0; d < D; ++d) xj[d] = ul[rows[k] * D + d];
#pragma unroll
            for (int di = 0; di < D; ++di)
#pragma unroll
              for (int dj = 0; dj < D; ++dj) acc[di] += m[di * D + dj][k] * xj[dj];
          }
        };
        auto load = [&](int32_t q, V (&m)[D * D]) {
#pragma unroll
          for (int k = 0; k < D * D; ++k) m[k] = *reinterpret_cast<const V*>(vit + (int64_t)k * a.nnzb_it + q);
        };
        int32_t q = team_here(rs[ps]) + lane * W;
        if (q < re[ps]) {
          if constexpr (kRes) {
            step(cv[ps], av[ps]);
          } else {
            V m[D * D];
            load(q, m);
            step(cv[ps], m);
          }
          for (q += GV * W; q < re[ps]; q += GV * W) {
            const I cols = *reinterpret_cast<const I*>(a.bcol_it + q);
            I rows;
#pragma unroll
            for (int k = 0; k < W; ++k) rows[k] = local_row(cols[k]);
            V m[D * D];
            load(q, m);
            step(rows, m);
          }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) acc[d] = group_sum<GV>(acc[d]);
        in_registers(acc);
        int64_t k;
        if (own(ps, k)) {
          wk[ps] = pick<T, D>(acc, lane);
          const double ud = uk[ps], rd = rk[ps];
          v3[0] += rd * ud;
          v3[1] += (double)wk[ps] * ud;
          v3[2] += rd * rd;
        }
      }
      if constexpr (CO) {
        coarse_rows(wk);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          v3[k] = wave_sum(v3[k]);
          if (wl == 0) s_red[sub][k][wid] = v3[k];
        }
        __syncthreads();
        if (!coarse_meet(true)) { alive = false; break; }
        if (threadIdx.x == 0) {
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            v3[k] = 0.0;
            for (int q = 0; q < kWaves; ++q) v3[k] += s_sum[k][q];
          }
          cg_scalars(&st, cg_in(&st), v3, it == a.chunk - 1);
          if constexpr (kFresh) {
            s_top = fmax(s_top, v3[2]);
            s_fresh = v3[2] < kTeamFresh * s_top;
            if (s_fresh) s_top = v3[2];
          }
        }
        coarse_apply_rows(yc);
      } else {
        if (!exchange_dots(v3)) { alive = false; break; }
        if (threadIdx.x == 0) cg_scalars(&st, cg_in(&st), v3, it == a.chunk - 1);
      }
      __syncthreads();
      if (st.done || st.need_ru) break;
    }
  }
  if (!alive && threadIdx.x == 0) team_give_up(a.abort, fits ? 1 : 2);
  // x is what the solve has reached, also after an aborted wait (the host continues from it)
#pragma unroll
  for (int ps = 0; ps < kPasses; ++ps) {
    int64_t k;
    if (own(ps, k)) a.x[caller(ps, k)] = xk[ps];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.st = st;
}

}  // namespace
