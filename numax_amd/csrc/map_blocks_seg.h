// map_blocks' structure-of-arrays solves for 8 < n <= 64, instantiated for
// double and float in map_blocks_f64.hip and map_blocks_f32.hip (one type a
// file: each of the unrolled kernels takes several seconds to compile).
#pragma once

#include <math.h>

#include "nmx_internal.h"

// every a - b * c below is a multiply, then a subtraction: numax's loops
// round twice
#pragma clang fp contract(off)

int map_blocks_seg(nmx_ctx* ctx, int kind, int n, int64_t batch, const double* xs, double* ys);
int map_blocks_seg(nmx_ctx* ctx, int kind, int n, int64_t batch, const float* xs, float* ys);

namespace {

template <typename T>
__device__ __forceinline__ T guard(T x) {  // guard_nonzero(x, 1e-30), numax/core/numeric.mojo:346-364
  const T f = (T)1e-30;
  const T m = fabs(x);
  return (m >= f || m != m) ? x : copysign(f, x);
}

// A segment of 16, 32 or 64 lanes per problem: lane i of a segment holds row i of A and b_i in registers (NP columns, n
// padded up).  The elimination is right-looking: every entry takes the same
// products in the same ascending order as numax's loops, so results are the
// oracle's bit for bit.  Rows are never moved: each lane keeps the position
// its row has in numax's swapped matrix, and the pivot row reaches the other
// lanes through a small LDS buffer of the wavefront's own.  b is carried
// along as one more column (the forward substitution's products in their own
// order); the back substitution's products u_ij x_j replace u_ij as each x_j
// appears, and row i's chain of subtractions runs on every lane at once.
//
// What bounds it: instruction issue -- an IEEE division a step in both
// sweeps, the multiply and the subtraction of every entry, and the back
// substitution's n^2/2 dependent subtractions that numax's order asks for.
// The batch is the fastest axis in memory, so a workgroup takes kProblems
// neighbouring problems and stages their entries through LDS in pieces of
// four columns: every global access is a run of 16 (or 8) problems.  A
// wavefront per problem with the matrix in LDS, which this replaces, read
// 8 bytes of each 128-byte line and walked the back substitution on one lane.
// 100,000 FP64 systems of order 24: 4.99 ms -> 0.56 ms (9.0x; 0.9 TB/s of the
// 4.8 TB/s a copy reaches).
template <int CTRL, typename T>
__device__ __forceinline__ T dpp_mov(T v) {
  if constexpr (sizeof(T) == 8) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xF, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
  } else {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
  }
}
// max over each segment of SEG lanes, in every lane of it
template <int SEG, typename T>
__device__ __forceinline__ T seg_max(T v) {
  v = fmax(v, dpp_mov<0xB1>(v));   // quad_perm 1,0,3,2
  v = fmax(v, dpp_mov<0x4E>(v));   // quad_perm 2,3,0,1
  v = fmax(v, dpp_mov<0x141>(v));  // row_half_mirror
  v = fmax(v, dpp_mov<0x140>(v));  // row_mirror
  if constexpr (SEG >= 32) v = fmax(v, __shfl_xor(v, 16));
  if constexpr (SEG >= 64) v = fmax(v, __shfl_xor(v, 32));
  return v;
}
template <int SEG>
__device__ __forceinline__ int seg_min(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, false));
  if constexpr (SEG >= 32) v = min(v, __shfl_xor(v, 16));
  if constexpr (SEG >= 64) v = min(v, __shfl_xor(v, 32));
  return v;
}

// One elimination step.  row: this segment's LDS buffer, NP + 1 entries.
template <int K, typename T, int NP, int SEG, int KIND>
__device__ __forceinline__ void seg_step(T (&m)[NP], T& v, int& pos, int i, T* row) {
  if constexpr (KIND == 1) {
    // cholesky (_array/cholesky.mojo:26-58) and forward_substitution: the
    // diagonal's root, then column k of L and x_k in one division
    const bool diag = i == K;
    if (diag) row[NP] = sqrt(guard(m[K]));
    wave_lds_order();
    const T ljj = row[NP];
    const T num = m[K], vk = v;
    const T q = (diag ? vk : num) / (diag ? guard(ljj) : ljj);
    if (i < NP) row[i] = q;  // lane K: x_k; the others l_ik (rows above k: unused)
    wave_lds_order();
    const T xk = row[K];
    if (i > K) {
      m[K] = q;
      v = v - q * xk;
#pragma unroll
      for (int j = K + 1; j < NP; j++) m[j] = m[j] - q * row[j];
    } else if (diag) {
      // row k of L^T, for the back substitution
      m[K] = ljj;
      v = xk;
#pragma unroll
      for (int j = K + 1; j < NP; j++) m[j] = row[j];
    }
    wave_lds_order();
  } else {
    bool piv = i == K;
    if constexpr (KIND == 0) {
      // the first largest |a_ik| from the diagonal down; a NaN on the
      // diagonal stays, a NaN below never wins
      const bool live = pos >= K;
      T mag = fabs(m[K]);
      if (mag != mag) mag = pos == K ? (T)INFINITY : (T)-1;
      mag = live ? mag : (T)-1;
      const bool hit = mag == seg_max<SEG>(mag) && live;
      const int pb = seg_min<SEG>(hit ? pos : 255);
      piv = hit && pos == pb;
      pos = piv ? K : (pos == K ? pb : pos);
    }
    if (piv) {
#pragma unroll
      for (int j = K; j < NP; j++) row[j] = m[j];
      row[NP] = v;
    }
    wave_lds_order();
    const bool below = KIND == 0 ? pos > K : i > K;
    if (below) {
      const T f = m[K] / guard(row[K]);
      v = v - f * row[NP];
#pragma unroll
      for (int j = K + 1; j < NP; j++) m[j] = m[j] - f * row[j];
    }
    wave_lds_order();
  }
}

template <int K, typename T, int NP, int SEG, int KIND>
__device__ __forceinline__ void seg_steps(T (&m)[NP], T& v, int& pos, int i, T* row, int n) {
  if constexpr (K < NP) {
    if (K < n) seg_step<K, T, NP, SEG, KIND>(m, v, pos, i, row);  // uniform
    seg_steps<K + 1, T, NP, SEG, KIND>(m, v, pos, i, row, n);
  }
}

// back_substitution (_array/triangular.mojo:46-63): row i subtracts u_ij x_j
// for j = i+1 .. n-1 in that order.  m[j] already holds u_ij x_j for j > I.
template <int I, typename T, int NP>
__device__ __forceinline__ void seg_back(T (&m)[NP], T v, int pos, T* x, int n) {
  if constexpr (I >= 0) {
    if (I < n) {  // uniform
      T total = v;
#pragma unroll
      for (int j = I + 1; j < NP; j++) total = total - m[j];
      const T q = total / guard(m[I]);
      if (pos == I) x[I] = q;
      wave_lds_order();
      m[I] = m[I] * x[I];
    }
    seg_back<I - 1, T, NP>(m, v, pos, x, n);
  }
}

template <int NP>
constexpr int seg_lanes() { return NP <= 16 ? 16 : NP <= 32 ? 32 : 64; }
template <int NP>
constexpr int seg_problems() { return NP <= 32 ? 16 : 8; }
template <int NP>
constexpr int seg_threads() { return seg_problems<NP>() * seg_lanes<NP>(); }

constexpr int kSegCols = 4;  // columns staged at a time

template <int J0, int C, typename T, int NP, int P, int NR>
__device__ __forceinline__ void seg_take(T (&m)[NP], T& v, int n, int q, int i, T (&stage)[kSegCols][P][NR]) {
  if constexpr (C < kSegCols) {
    constexpr int J = J0 + C;
    const T val = J <= n && i < n ? stage[C][q][i] : (T)0;
    if constexpr (J < NP) m[J] = J < n ? val : (T)0;
    if (J == n) v = val;
    seg_take<J0, C + 1>(m, v, n, q, i, stage);
  }
}

// Columns J0 .. J0+3 (column n is b) of the workgroup's problems through LDS
// into the owning lanes' registers, then the next four.
template <int J0, typename T, int NP, int P, int NR>
__device__ __forceinline__ void seg_stage(T (&m)[NP], T& v, int n, int64_t batch, const T* __restrict__ xs, int64_t lp,
                                          int lq, int lr, int q, int i, T (&stage)[kSegCols][P][NR]) {
  if constexpr (J0 <= NP) {
    if (J0 <= n) {  // uniform
      for (int e = lr; e < n * kSegCols; e += seg_threads<NP>() / P) {
        const int r = e / kSegCols, j = J0 + e % kSegCols;
        T val = 0;
        if (j < n) val = xs[(int64_t)(r * n + j) * batch + lp];
        else if (j == n) val = xs[(int64_t)(n * n + r) * batch + lp];
        stage[e % kSegCols][lq][r] = val;
      }
      __syncthreads();
    }
    seg_take<J0, 0>(m, v, n, q, i, stage);
    if (J0 <= n) __syncthreads();
    seg_stage<J0 + kSegCols>(m, v, n, batch, xs, lp, lq, lr, q, i, stage);
  }
}

template <typename T, int NP, int KIND>
__global__ void __launch_bounds__(seg_threads<NP>()) __attribute__((amdgpu_waves_per_eu(NP <= 32 ? 4 : 2)))
map_blocks_seg_kernel(int n, int64_t batch,
                                                                           const T* __restrict__ xs,
                                                                           T* __restrict__ ys) {
  constexpr int SEG = seg_lanes<NP>(), P = seg_problems<NP>(), NT = seg_threads<NP>();
  constexpr int NR = NP | 1;   // odd: neighbouring problems fall in different banks
  __shared__ T stage[kSegCols][P][NR];
  __shared__ __attribute__((aligned(16))) T rows[P][NP + 4];
  const int t = threadIdx.x;
  const int q = t / SEG, i = t % SEG;     // this thread's problem and row
  const int lq = t % P, lr = t / P;       // staging: problem, then (row, column)
  const int64_t p0 = (int64_t)blockIdx.x * P;
  const int64_t lp = min(p0 + lq, batch - 1);  // past the end: any valid problem, not stored
  T m[NP], v = 0;
  seg_stage<0>(m, v, n, batch, xs, lp, lq, lr, q, i, stage);
  int pos = i;
  T* row = rows[q];
  seg_steps<0, T, NP, SEG, KIND>(m, v, pos, i, row, n);
  // padded columns: whatever an infinite multiplier left there
#pragma unroll
  for (int j = 9; j < NP; j++) m[j] = j < n ? m[j] : (T)0;
  seg_back<NP - 1, T, NP>(m, v, pos, row, n);
  __syncthreads();
  for (int e = lr; e < n; e += NT / P)
    if (p0 + lq < batch) ys[(int64_t)e * batch + p0 + lq] = rows[lq][e];
}

template <typename T, int NP>
int map_blocks_seg_launch(nmx_ctx* ctx, int kind, int n, int64_t batch, const T* xs, T* ys) {
  const int64_t P = seg_problems<NP>();
  const unsigned grid = (unsigned)((batch + P - 1) / P);
  constexpr int NT = seg_threads<NP>();
  if (kind == 0) map_blocks_seg_kernel<T, NP, 0><<<grid, NT, 0, ctx->stream>>>(n, batch, xs, ys);
  if (kind == 1) map_blocks_seg_kernel<T, NP, 1><<<grid, NT, 0, ctx->stream>>>(n, batch, xs, ys);
  if (kind == 2) map_blocks_seg_kernel<T, NP, 2><<<grid, NT, 0, ctx->stream>>>(n, batch, xs, ys);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

// the narrowest padding of n: instructions go with NP^2, registers with NP
template <typename T>
int map_blocks_seg_any(nmx_ctx* ctx, int kind, int n, int64_t batch, const T* xs, T* ys) {
  if (n <= 16) return map_blocks_seg_launch<T, 16>(ctx, kind, n, batch, xs, ys);
  if (n <= 24) return map_blocks_seg_launch<T, 24>(ctx, kind, n, batch, xs, ys);
  if (n <= 32) return map_blocks_seg_launch<T, 32>(ctx, kind, n, batch, xs, ys);
  if (n <= 48) return map_blocks_seg_launch<T, 48>(ctx, kind, n, batch, xs, ys);
  return map_blocks_seg_launch<T, 64>(ctx, kind, n, batch, xs, ys);
}

}  // namespace
