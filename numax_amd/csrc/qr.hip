// Blocked Householder QR, FP64 and FP32, device-resident: numax's Tensor-tier
// qr_factor / QR.apply_q_transpose / QR.q / QR.r / QR.solve / lstsq
// (numax/linalg/qr.mojo:330-821).
//
// Right-looking and blocked as numax's: a `block`-wide panel of reflectors
// is factored in place (geqr2_panel, numax/linalg/panel.mojo:1975-2073,
// LAPACK dlarfg's convention), then its block reflector reaches everything
// to its right at once as C -= V (T^T (V^T C)) (qr.mojo:123-327) with T
// the forward columnwise triangular factor (larft_panel, panel.mojo:
// 2076-2169).  The three products are the library's MFMA GEMM; the panel
// is one workgroup of 16 wavefronts streaming the panel's rows, one column
// at a time: the column norm and the panel's dot products are workgroup
// reductions (shuffles within a wavefront, LDS across them).  T is built
// from the Gram matrix V^T V, itself one GEMM of an explicit V (unit
// diagonal, zeros above), which the three block-reflector products use too.
// Panels of at most 16 columns, numax's default width, take two launches each
// instead: a register panel that leaves T too, and one fused application.
// lstsq of 2500 x 300 FP32: 21.3 ms -> 1.8 ms.
#include <math.h>

#include "tile16.h"

namespace {

constexpr int kQrMaxBlock = 64;  // panel width the kernels take
constexpr int kQrThreads = 1024;
constexpr int kQrWaves = kQrThreads / 64;
constexpr int kQrChunk = 16;     // panel columns whose dot products are reduced together

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

// Sum over the workgroup of NV values per thread; every thread gets the totals.
template <typename T, int NV>
__device__ __forceinline__ void block_sum(T (&v)[NV], T (*red)[kQrChunk], T* out) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
  for (int u = 0; u < NV; u++) {
    const T s = wave_sum(v[u]);
    if (lane == 0) red[w][u] = s;
  }
  __syncthreads();
  if (t < NV) {
    T s = 0;
    for (int q = 0; q < kQrWaves; q++) s += red[q][t];
    out[t] = s;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NV; u++) v[u] = out[u];
  __syncthreads();
}

// geqr2_panel on A[k:m, k:k+nb] in place, tau[k..k+nb).  Per column: sigma =
// sum of squares below the diagonal; sigma == 0 leaves the column and gives
// tau = 0; otherwise beta = -sign(alpha) sqrt(alpha^2 + sigma), tau =
// (beta - alpha) / beta, v = x / (alpha - beta) below the diagonal, R_kk =
// beta, and each later panel column c gets c -= tau (c_k + v^T c_below) v.
template <typename T>
__global__ void __launch_bounds__(kQrThreads) geqr2_kernel(int m, T* __restrict__ A, int lda, T* __restrict__ tau,
                                                           int k, int nb) {
  __shared__ T red[kQrWaves][kQrChunk];
  __shared__ T tot[kQrChunk];
  const int t = threadIdx.x;
  for (int j = 0; j < nb; j++) {
    const int col = k + j;
    T s[1] = {T(0)};
    for (int i = col + 1 + t; i < m; i += kQrThreads) {
      const T a = A[(int64_t)i * lda + col];
      s[0] += a * a;
    }
    block_sum<T, 1>(s, red, tot);
    const T sigma = s[0];
    const T alpha = A[(int64_t)col * lda + col];
    if (sigma == T(0)) {
      if (t == 0) tau[col] = T(0);
      continue;
    }
    T beta = sqrt(alpha * alpha + sigma);
    if (alpha > T(0)) beta = -beta;
    const T tj = (beta - alpha) / beta;
    const T scale = T(1) / (alpha - beta);
    for (int i = col + 1 + t; i < m; i += kQrThreads) A[(int64_t)i * lda + col] *= scale;
    __syncthreads();  // the scaled column and R_kk before any thread reads them back
    if (t == 0) {
      A[(int64_t)col * lda + col] = beta;
      tau[col] = tj;
    }
    for (int c0 = j + 1; c0 < nb; c0 += kQrChunk) {
      T d[kQrChunk];
#pragma unroll
      for (int u = 0; u < kQrChunk; u++) d[u] = T(0);
      for (int i = col + 1 + t; i < m; i += kQrThreads) {
        const T* row = A + (int64_t)i * lda;
        const T v = row[col];
#pragma unroll
        for (int u = 0; u < kQrChunk; u++)
          if (c0 + u < nb) d[u] += v * row[k + c0 + u];
      }
      block_sum<T, kQrChunk>(d, red, tot);
      // dot_c = c_k + v^T c_below: the unit entry of v meets row col
      T f[kQrChunk];
#pragma unroll
      for (int u = 0; u < kQrChunk; u++)
        f[u] = c0 + u < nb ? tj * (A[(int64_t)col * lda + k + c0 + u] + d[u]) : T(0);
      __syncthreads();  // row col read by every thread before it is rewritten
      if (t < kQrChunk && c0 + t < nb) {
        T* p = A + (int64_t)col * lda + k + c0 + t;
        *p -= tj * (*p + tot[t]);
      }
      for (int i = col + 1 + t; i < m; i += kQrThreads) {
        T* row = A + (int64_t)i * lda;
        const T v = row[col];
#pragma unroll
        for (int u = 0; u < kQrChunk; u++)
          if (c0 + u < nb) row[k + c0 + u] -= f[u] * v;
      }
      __syncthreads();
    }
  }
}

// V (rows x nb, ld nb) explicit from the panel: unit diagonal, zeros above.
template <typename T>
__global__ void explicit_v_kernel(int rows, int nb, const T* __restrict__ A, int lda, int k, T* __restrict__ V) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)rows * nb) return;
  const int r = (int)(idx / nb), c = (int)(idx % nb);
  V[idx] = r == c ? T(1) : (r > c ? A[(int64_t)(k + r) * lda + k + c] : T(0));
}

// larft_panel's T (forward, columnwise, upper, nb x nb) from the Gram matrix
// G = V^T V and tau: T_ii = tau_i, T[0:i, i] = -tau_i T[0:i, 0:i] G[0:i, i].
template <typename E>
__global__ void __launch_bounds__(64) larft_kernel(int nb, const E* __restrict__ G, const E* __restrict__ tau, int k,
                                                   E* __restrict__ T) {
  __shared__ E Ts[kQrMaxBlock][kQrMaxBlock + 1];
  __shared__ E g[kQrMaxBlock];
  const int q = threadIdx.x;
  for (int r = 0; r < nb; r++)
    if (q < nb) Ts[r][q] = E(0);
  if (q == 0) Ts[0][0] = tau[k];
  __syncthreads();
  for (int i = 1; i < nb; i++) {
    const E ti = tau[k + i];
    if (q < i) g[q] = -ti * G[q * nb + i];
    __syncthreads();
    E s = E(0);
    if (q < i)
      for (int r = q; r < i; r++) s += Ts[q][r] * g[r];
    __syncthreads();
    if (q < i) Ts[q][i] = s;
    if (q == 0) Ts[i][i] = ti;
    __syncthreads();
  }
  for (int r = 0; r < nb; r++)
    if (q < nb) T[r * nb + q] = Ts[r][q];
}

template <typename T>
__global__ void identity_kernel(int m, int n, T* __restrict__ Q, int ldq) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int r = (int)(idx / n), c = (int)(idx % n);
  Q[(int64_t)r * ldq + c] = r == c ? T(1) : T(0);
}

template <typename T>
__global__ void upper_kernel(int n, const T* __restrict__ A, int lda, T* __restrict__ R, int ldr) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * n) return;
  const int r = (int)(idx / n), c = (int)(idx % n);
  R[(int64_t)r * ldr + c] = r <= c ? A[(int64_t)r * lda + c] : T(0);
}

// Workspace of one block reflector: V (rows x nb), G and T (nb x nb), W and Y
// (nb x width), carved from the context workspace.
template <typename T>
struct Reflector {
  T* V;
  T* G;
  T* T_;
  T* W;
  T* Y;
};

template <typename T>
size_t reflector_bytes(int m, int nb, int width) {
  const size_t e = (size_t)m * nb + 2 * (size_t)nb * nb + 2 * (size_t)nb * (width > 0 ? width : 1);
  return e * sizeof(T);
}

template <typename T>
Reflector<T> carve(void* ws, int m, int nb, int width) {
  Reflector<T> r;
  r.V = (T*)ws;
  r.G = r.V + (size_t)m * nb;
  r.T_ = r.G + (size_t)nb * nb;
  r.W = r.T_ + (size_t)nb * nb;
  r.Y = r.W + (size_t)nb * (width > 0 ? width : 1);
  return r;
}

// V and T of the panel at column k (nb wide) of the m x n factored matrix.
template <typename T>
int build_reflector(nmx_ctx* ctx, const Reflector<T>& w, int m, const T* QR, int lda, const T* tau, int k, int nb) {
  const int rows = m - k;
  explicit_v_kernel<T><<<(unsigned)(((int64_t)rows * nb + 255) / 256), 256, 0, ctx->stream>>>(rows, nb, QR, lda, k,
                                                                                             w.V);
  NMX_HIP(ctx, hipGetLastError());
  NMX_TRY(gemm_launch<T>(ctx, 1, 0, nb, nb, rows, T(1), w.V, nb, w.V, nb, T(0), w.G, nb));
  larft_kernel<T><<<1, 64, 0, ctx->stream>>>(nb, w.G, tau, k, w.T_);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

// C (rows x width, ld ldc; rows = m - k) := (I - V op(T) V^T) C, op(T) = T^T
// when `trans` (Q^T, the factorization's and apply_q_transpose's direction),
// T otherwise (Q, QR.q's).
template <typename T>
int apply_reflector(nmx_ctx* ctx, const Reflector<T>& w, int rows, int nb, int width, int trans, T* C, int ldc) {
  if (width <= 0) return NMX_OK;
  NMX_TRY(gemm_launch<T>(ctx, 1, 0, nb, width, rows, T(1), w.V, nb, C, ldc, T(0), w.W, width));
  NMX_TRY(gemm_launch<T>(ctx, trans, 0, nb, width, nb, T(1), w.T_, nb, w.W, width, T(0), w.Y, width));
  return gemm_launch<T>(ctx, 0, 0, rows, width, nb, T(-1), w.V, nb, w.Y, width, T(1), C, ldc);
}

// ---- panels of at most 16 columns (numax's default width) --------------------
//
// The panel in registers: a thread holds R rows of one column (c = lane % 16),
// so the reflector's column reaches the other columns of its rows as a DPP
// broadcast inside a 16-lane row, and one value per column crosses the row
// groups of a step.  What bounds it is the chain of steps (two sums' worth of
// multiply-adds, one LDS round and barrier, a root and two divisions); the
// streaming kernel above walked the panel in memory three times a column.
// 2500 x 16 FP32: 627 us -> 41 us.  T comes with it: a step's sums over the
// finished columns are the V^T v_K that larft_panel (panel.mojo:2076-2169)
// builds it from.
constexpr int kNarrow = 16;

template <typename T, int NW>
struct PanelLds {
  T part[2][NW][kNarrow];  // column sums by wavefront
  T row[2][kNarrow];       // row K of the panel
  T G[kNarrow][kNarrow];   // G[K][c] = v_c^T v_K, c < K
  T tau[kNarrow];
};

// Reflector K: x = column K below its diagonal, sigma = x^T x, and for every
// later column A_c -= tau (A_Kc + scale x^T A_c) [1; scale x] -- geqr2_panel's
// dlarfg convention.  Row K leaves the registers (zero there) before the sums,
// so sums over all rows are sums below the diagonal.  x stays unscaled in the
// registers; lane K keeps the column's scale in `sc`.
template <int K, typename T, int R, int NW>
__device__ __forceinline__ void panel_step(T (&a)[R], T& sc, int t, int nb, T* __restrict__ A, int lda,
                                           T* __restrict__ tau, PanelLds<T, NW>& L) {
  constexpr int buf = K & 1;
  asm volatile("" : "+v"(t));  // the lane masks below are made here, not kept over the steps
  const int lane = t & 63, wave = t >> 6, c = lane & 15;
  if (t < kNarrow) {
    L.row[buf][c] = a[K] * sc;
    a[K] = T(0);
  }
  T p0 = 0, p1 = 0, p2 = 0, p3 = 0;
#pragma unroll
  for (int r = 0; r < R; r += 4)
    fmac_bcast4<K>(p0, p1, p2, p3, a[r], a[r + 1], a[r + 2], a[r + 3], a[r], a[r + 1], a[r + 2], a[r + 3]);
  T p = (p0 + p1) + (p2 + p3);
  p += __shfl_xor(p, 16);
  p += __shfl_xor(p, 32);
  if (lane < kNarrow) L.part[buf][wave][c] = p;
  __syncthreads();
  T tot = 0;
#pragma unroll
  for (int w = 0; w < NW; w++) tot += L.part[buf][w][c];
  const T rk = L.row[buf][c];
  const T sigma = row_bcast<K>(tot), alpha = row_bcast<K>(rk);
  T beta = sqrt(alpha * alpha + sigma);
  if (alpha > T(0)) beta = -beta;
  const bool none = sigma == T(0);
  const T tj = none ? T(0) : (beta - alpha) / beta;
  const T scale = none ? T(0) : T(1) / (alpha - beta);
  // v_K^T A_c; for finished columns v_K^T v_c.  Of a column that is zero below
  // its diagonal v_K is a unit vector: nothing below it counts, infinities included
  const T g = none ? rk : rk + scale * tot * sc;
  const T f = c > K && !none ? tj * g : T(0);
  const T nfs = -(f * scale);
  if (c == K && !none) sc = scale;
  if (c >= K) {  // lane K, which the products read, is among them; its own is 0
#pragma unroll
    for (int r = 0; r < R; r += 4) fmac_self4<K>(a[r], a[r + 1], a[r + 2], a[r + 3], nfs);
  }
  if (t < kNarrow) {
    if (c < K) L.G[K][c] = g;
    // row K of the result: V left of the diagonal, R from it on
    if (c < nb) A[(int64_t)K * lda + c] = c == K ? (none ? alpha : beta) : rk - f;
    if (c == K) {
      tau[K] = tj;
      L.tau[K] = tj;
    }
  }
}

// T (16 x 16, row-major) by lanes 0..15 of a wavefront, lane r row r:
// T_ii = tau_i, T[0:i, i] = -tau_i T[0:i, 0:i] (V^T v_i).
template <typename T>
__device__ __forceinline__ void narrow_t(int nb, const T (&G)[kNarrow][kNarrow], const T* tau, int r, T* out) {
  T row[kNarrow];
#pragma unroll
  for (int i = 0; i < kNarrow; i++) {
    T s = 0;
#pragma unroll
    for (int q = 0; q < i; q++) s += row[q] * G[i][q];  // row[q] = 0 left of the diagonal
    const T ti = i < nb ? tau[i] : T(0);
    row[i] = i >= nb || i < r ? T(0) : (i == r ? ti : -ti * s);
  }
#pragma unroll
  for (int i = 0; i < kNarrow; i++) out[r * kNarrow + i] = row[i];
}

template <int K, typename T, int R, int NW>
__device__ __forceinline__ void panel_steps(T (&a)[R], T& sc, int t, int nb, T* A, int lda, T* tau, PanelLds<T, NW>& L) {
  if constexpr (K < kNarrow) {
    if (K < nb) panel_step<K, T, R, NW>(a, sc, t, nb, A, lda, tau, L);  // uniform
    panel_steps<K + 1, T, R, NW>(a, sc, t, nb, A, lda, tau, L);
  }
}

// A: the panel's top left corner, rows x nb with rows <= 4 NW R.
template <typename T, int R, int NW>
__global__ void __launch_bounds__(64 * NW) geqr2_narrow_kernel(int rows, int nb, T* __restrict__ A, int lda,
                                                               T* __restrict__ tau, T* __restrict__ Tout) {
  __shared__ PanelLds<T, NW> L;
  const int t = threadIdx.x, c = t & 15, row0 = (t >> 4) * R;
  T a[R];
  const T* src = A + (int64_t)row0 * lda + c;
#pragma unroll
  for (int r = 0; r < R; r++) a[r] = (row0 + r < rows) & (c < nb) ? src[(int64_t)r * lda] : T(0);
  if (t < kNarrow)
    for (int i = 0; i < kNarrow; i++) L.G[t][i] = T(0);
  __syncthreads();  // and every load is done before row 0 is stored
  T sc = T(1);  // a finished column's reflector is its x times this
  panel_steps<0, T, R, NW>(a, sc, t, nb, A, lda, tau, L);
  T* dst = A + (int64_t)row0 * lda + c;
#pragma unroll
  for (int r = 0; r < R; r++)
    if ((row0 + r < rows) & (c < nb) & (row0 + r >= nb)) dst[(int64_t)r * lda] = a[r] * sc;
  if (t < kNarrow) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    narrow_t<T>(nb, L.G, L.tau, t, Tout);
  }
}

// V[r][i] of a narrow panel at A (unit diagonal, zeros above it and past nb)
template <typename T>
__device__ __forceinline__ T narrow_v(const T* __restrict__ A, int lda, int rows, int nb, int r, int i) {
  if (r < i || i >= nb || r >= rows) return T(0);
  return r == i ? T(1) : A[(int64_t)r * lda + i];
}

// T of panels k = 0, 16.. of an already factored matrix, one workgroup each.
template <typename T>
__global__ void __launch_bounds__(kQrThreads) narrow_t_kernel(int m, int n, int block, const T* __restrict__ QR, int lda,
                                                              const T* __restrict__ tau, T* __restrict__ Tout) {
  __shared__ T part[kQrWaves][kNarrow][kNarrow];
  __shared__ T G[kNarrow][kNarrow];
  __shared__ T tl[kNarrow];
  const int k = blockIdx.x * block, nb = min(block, n - k), rows = m - k;
  const T* A = QR + (int64_t)k * lda + k;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  typename Acc<T>::type acc = {0, 0, 0, 0};
  for (int r0 = 16 * w; r0 < rows; r0 += 16 * kQrWaves) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const T v = narrow_v<T>(A, lda, rows, nb, r0 + acc_row<T>(lane, e), lane & 15);
      acc = mma(v, v, acc);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; e++) part[w][acc_row<T>(lane, e)][lane & 15] = acc[e];
  if (t < kNarrow) tl[t] = t < nb ? tau[k + t] : T(0);
  __syncthreads();
  if (t < 256) {
    T s = 0;
    for (int q = 0; q < kQrWaves; q++) s += part[q][t >> 4][t & 15];
    G[t >> 4][t & 15] = s;
  }
  __syncthreads();
  if (t < kNarrow) narrow_t<T>(nb, G, tl, t, Tout + (int64_t)blockIdx.x * kNarrow * kNarrow);
}

// Tiles of 16 rows, wavefront w every 16th: the first and a last partial one
// with every element's place looked at, the full ones below the unit triangle
// four at a time, so that their loads are in flight together.
template <typename F>
__device__ __forceinline__ void walk_tiles(int rows, int w, F&& tile) {
  int r0 = 16 * w;
  if (r0 == 0) {
    tile(0, false);
    r0 = 16 * kQrWaves;
  }
#pragma unroll 4
  for (; r0 + 16 <= rows; r0 += 16 * kQrWaves) tile(r0, true);
  if (r0 < rows) tile(r0, false);
}

// C := (I - V op(T) V^T) C for a panel of at most 16 reflectors, 16 columns of
// C a workgroup, in one launch: W = V^T C over all rows on MFMA (each wavefront
// every 16th tile of 16 rows), the wavefronts' W summed in order through LDS,
// Y = op(T) W by 256 threads, then C -= V Y on a second walk down the rows,
// whose 16 columns are still in L2.  op(T) = T^T when `trans`.  The last
// columns of the grid belong to a second matrix (lstsq's right-hand sides).
// What bounds it is the latency of the two walks.  As three products of the
// general GEMM the first one, one tile wide, ran 2500 rows deep on five
// workgroups: 63 us against 30 us for this whole launch at 2500 x 284.
template <typename T>
__global__ void __launch_bounds__(kQrThreads) narrow_apply_kernel(int rows, int nb, const T* __restrict__ A, int lda,
                                                                  const T* __restrict__ Tm, int trans, T* __restrict__ C1,
                                                                  int ldc1, int width1, T* __restrict__ C2, int ldc2,
                                                                  int width2) {
  typedef typename Acc<T>::type acc_t;
  __shared__ T part[kQrWaves][kNarrow][kNarrow];
  __shared__ T W[kNarrow][kNarrow], Y[kNarrow][kNarrow];
  const int tiles1 = (width1 + 15) / 16;
  const bool second = (int)blockIdx.x >= tiles1;
  T* C = second ? C2 : C1;
  const int ldc = second ? ldc2 : ldc1, width = second ? width2 : width1;
  const int j0 = 16 * ((int)blockIdx.x - (second ? tiles1 : 0));
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int lc = lane & 15, lk = lane >> 4;
  const bool in = j0 + lc < width;
  C += j0 + (in ? lc : 0);
  acc_t acc = {0, 0, 0, 0};
  const int vc = min(lc, nb - 1);
  walk_tiles(rows, w, [&](int r0, bool full) {
    T v[4], cv[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = r0 + acc_row<T>(lane, e);
      v[e] = full ? A[(int64_t)r * lda + vc] : narrow_v<T>(A, lda, rows, nb, r, lc);
      cv[e] = full || r < rows ? C[(int64_t)r * ldc] : T(0);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) acc = mma(lc < nb ? v[e] : T(0), cv[e], acc);
  });
#pragma unroll
  for (int e = 0; e < 4; e++) part[w][acc_row<T>(lane, e)][lc] = acc[e];
  __syncthreads();
  if (t < 256) {
    T s = 0;
#pragma unroll
    for (int q = 0; q < kQrWaves; q++) s += part[q][t >> 4][t & 15];
    W[t >> 4][t & 15] = s;
  }
  __syncthreads();
  if (t < 256) {
    const int i = t >> 4, j = t & 15;
    T s = 0;
#pragma unroll
    for (int q = 0; q < kNarrow; q++) s += (trans ? Tm[q * kNarrow + i] : Tm[i * kNarrow + q]) * W[q][j];
    Y[i][j] = s;
  }
  __syncthreads();
  T y[4];
#pragma unroll
  for (int q = 0; q < 4; q++) y[q] = Y[4 * lk + q][lc];
  walk_tiles(rows, w, [&](int r0, bool full) {
    T v[4], cv[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int i = 4 * lk + q;
      v[q] = full ? A[(int64_t)(r0 + lc) * lda + min(i, nb - 1)] : narrow_v<T>(A, lda, rows, nb, r0 + lc, i);
      if (i >= nb) v[q] = T(0);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = r0 + acc_row<T>(lane, e);
      cv[e] = full || r < rows ? C[(int64_t)r * ldc] : T(0);
    }
    acc_t d = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; q++) d = mma(v[q], y[q], d);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = r0 + acc_row<T>(lane, e);
      if (in && (full || r < rows)) C[(int64_t)r * ldc] = cv[e] - d[e];
    }
  });
}

template <typename T>
int narrow_apply(nmx_ctx* ctx, int rows, int nb, const T* A, int lda, const T* Tm, int trans, T* C1, int ldc1, int width1,
                 T* C2, int ldc2, int width2) {
  const int tiles = ceil_div(width1, 16) + ceil_div(width2, 16);
  if (tiles <= 0) return NMX_OK;
  ProfScope ps(ctx, K_GEMM, 4.0 * rows * nb * (double)(width1 + width2), 0.0);
  narrow_apply_kernel<T><<<tiles, kQrThreads, 0, ctx->stream>>>(rows, nb, A, lda, Tm, trans, C1, ldc1, width1, C2, ldc2,
                                                                width2);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

// Factors the panel at A (rows x nb, nb <= 16) and leaves its T in Tm.  The
// register kernels hold 4 NW R rows; the fewest that fit, since a step's sums
// go with R and its LDS round with NW.  A taller panel streams through memory.
template <typename T>
int narrow_panel(nmx_ctx* ctx, int m, int k, int nb, T* A, int lda, T* tau, T* Tm) {
  const int rows = m - k;
  T* P = A + (int64_t)k * lda + k;
  ProfScope ps(ctx, K_QR_PANEL, 4.0 * (double)rows * nb * nb, 2.0 * sizeof(T) * (double)rows * nb);
  if (rows <= 256) geqr2_narrow_kernel<T, 16, 4><<<1, 256, 0, ctx->stream>>>(rows, nb, P, lda, tau + k, Tm);
  else if (rows <= 1024) geqr2_narrow_kernel<T, 16, 16><<<1, 1024, 0, ctx->stream>>>(rows, nb, P, lda, tau + k, Tm);
  else if (rows <= 2048) geqr2_narrow_kernel<T, 32, 16><<<1, 1024, 0, ctx->stream>>>(rows, nb, P, lda, tau + k, Tm);
  else if (sizeof(T) == 4 && rows <= 4096) {
    if constexpr (sizeof(T) == 4)
      geqr2_narrow_kernel<T, 64, 16><<<1, 1024, 0, ctx->stream>>>(rows, nb, P, lda, tau + k, Tm);
  } else {
    geqr2_kernel<T><<<1, kQrThreads, 0, ctx->stream>>>(m, A, lda, tau, k, nb);
    NMX_HIP(ctx, hipGetLastError());
    narrow_t_kernel<T><<<1, kQrThreads, 0, ctx->stream>>>(rows, nb, nb, P, lda, tau + k, Tm);
  }
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

// Blocked QR with panels of at most 16 columns; every panel's reflector also
// reaches B (m x nrhs; nrhs 0: none), which leaves Q^T B there.
template <typename T>
int geqrf_narrow(nmx_ctx* ctx, int m, int n, T* A, int lda, T* tau, int block, T* B, int ldb, int nrhs) {
  void* ws = nullptr;
  NMX_TRY(nmx_workspace(ctx, kNarrow * kNarrow * sizeof(T), &ws));
  for (int k = 0; k < n; k += block) {
    const int nb = std::min(block, n - k), width = n - k - nb;
    NMX_TRY(narrow_panel<T>(ctx, m, k, nb, A, lda, tau, (T*)ws));
    const T* P = A + (int64_t)k * lda + k;
    NMX_TRY(narrow_apply<T>(ctx, m - k, nb, P, lda, (const T*)ws, 1, A + (int64_t)k * lda + k + nb, lda, width,
                            B + (int64_t)k * ldb, ldb, nrhs));
  }
  return NMX_OK;
}

// The Ts of all panels of a factored matrix, in the context workspace.
template <typename T>
int narrow_all_t(nmx_ctx* ctx, int m, int n, const T* QR, int lda, const T* tau, int block, const T** out) {
  const int steps = ceil_div(n, block);
  void* ws = nullptr;
  NMX_TRY(nmx_workspace(ctx, (size_t)steps * kNarrow * kNarrow * sizeof(T), &ws));
  narrow_t_kernel<T><<<steps, kQrThreads, 0, ctx->stream>>>(m, n, block, QR, lda, tau, (T*)ws);
  NMX_HIP(ctx, hipGetLastError());
  *out = (const T*)ws;
  return NMX_OK;
}

template <typename T>
int geqrf_impl(nmx_ctx* ctx, int m, int n, T* A, int lda, T* tau, int block) {
  if (block <= kNarrow) return geqrf_narrow<T>(ctx, m, n, A, lda, tau, block, (T*)nullptr, 0, 0);
  void* ws = nullptr;
  NMX_TRY(nmx_workspace(ctx, reflector_bytes<T>(m, block, n), &ws));
  const Reflector<T> w = carve<T>(ws, m, block, n);
  for (int k = 0; k < n; k += block) {
    const int nb = std::min(block, n - k);
    {
      ProfScope ps(ctx, K_QR_PANEL, 4.0 * (double)(m - k) * nb * nb, 2.0 * sizeof(T) * (double)(m - k) * nb * nb);
      geqr2_kernel<T><<<1, kQrThreads, 0, ctx->stream>>>(m, A, lda, tau, k, nb);
      NMX_HIP(ctx, hipGetLastError());
    }
    if (k + nb < n) {
      NMX_TRY(build_reflector(ctx, w, m, A, lda, tau, k, nb));
      NMX_TRY(apply_reflector(ctx, w, m - k, nb, n - k - nb, 1, A + (int64_t)k * lda + k + nb, lda));
    }
  }
  return NMX_OK;
}

// B (m x nrhs) := Q^T B (trans) or Q B, panels in the order each needs.
template <typename T>
int ormqr_impl(nmx_ctx* ctx, int trans, int m, int n, int nrhs, const T* QR, int lda, const T* tau, T* B, int ldb,
               int block) {
  const int steps = ceil_div(n, block);
  if (block <= kNarrow) {
    const T* Tm = nullptr;
    NMX_TRY(narrow_all_t<T>(ctx, m, n, QR, lda, tau, block, &Tm));
    for (int s = 0; s < steps; s++) {
      const int p = trans ? s : steps - 1 - s, k = p * block;
      NMX_TRY(narrow_apply<T>(ctx, m - k, std::min(block, n - k), QR + (int64_t)k * lda + k, lda,
                              Tm + (size_t)p * kNarrow * kNarrow, trans, B + (int64_t)k * ldb, ldb, nrhs, (T*)nullptr, 0, 0));
    }
    return NMX_OK;
  }
  void* ws = nullptr;
  NMX_TRY(nmx_workspace(ctx, reflector_bytes<T>(m, block, nrhs), &ws));
  const Reflector<T> w = carve<T>(ws, m, block, nrhs);
  for (int s = 0; s < steps; s++) {
    const int k = (trans ? s : steps - 1 - s) * block;
    const int nb = std::min(block, n - k);
    NMX_TRY(build_reflector(ctx, w, m, QR, lda, tau, k, nb));
    NMX_TRY(apply_reflector(ctx, w, m - k, nb, nrhs, trans, B + (int64_t)k * ldb, ldb));
  }
  return NMX_OK;
}

int check_qr_args(nmx_ctx* ctx, int m, int n, int lda, int block) {
  if (!ctx) return -1;
  if (m < 0) return -2;
  if (n < 0 || n > m) return -3;
  if (lda < std::max(1, n)) return -5;
  if (block < 1 || block > kQrMaxBlock) return -7;
  return NMX_OK;
}

}  // namespace

namespace {

template <typename T>
int geqrf_api(nmx_ctx* ctx, int m, int n, T* A, int lda, T* tau, int block) {
  NMX_TRY(check_qr_args(ctx, m, n, lda, block));
  if (n == 0) return NMX_OK;
  if (!A) return -4;
  if (!tau) return -6;
  return geqrf_impl<T>(ctx, m, n, A, lda, tau, block);
}

template <typename T>
int ormqr_api(nmx_ctx* ctx, int trans, int m, int n, int nrhs, const T* QR, int lda, const T* tau, T* B, int ldb,
              int block) {
  if (!ctx) return -1;
  if (m < 0) return -3;
  if (n < 0 || n > m) return -4;
  if (nrhs < 0) return -5;
  if (lda < std::max(1, n)) return -7;
  if (ldb < std::max(1, nrhs)) return -10;
  if (block < 1 || block > kQrMaxBlock) return -11;
  if (n == 0 || nrhs == 0) return NMX_OK;
  if (!QR) return -6;
  if (!tau) return -8;
  if (!B) return -9;
  return ormqr_impl<T>(ctx, trans ? 1 : 0, m, n, nrhs, QR, lda, tau, B, ldb, block);
}

template <typename T>
int orgqr_api(nmx_ctx* ctx, int m, int n, const T* QR, int lda, const T* tau, T* Q, int ldq, int block) {
  NMX_TRY(check_qr_args(ctx, m, n, lda, block));
  if (ldq < std::max(1, n)) return -8;
  if (n == 0) return NMX_OK;
  if (!QR) return -4;
  if (!tau) return -6;
  if (!Q) return -7;
  identity_kernel<T><<<(unsigned)(((int64_t)m * n + 255) / 256), 256, 0, ctx->stream>>>(m, n, Q, ldq);
  NMX_HIP(ctx, hipGetLastError());
  // last panel first; columns left of the panel are unchanged (V^T e_j = 0)
  if (block <= kNarrow) {
    const T* Tm = nullptr;
    NMX_TRY(narrow_all_t<T>(ctx, m, n, QR, lda, tau, block, &Tm));
    for (int p = ceil_div(n, block) - 1; p >= 0; p--) {
      const int k = p * block;
      NMX_TRY(narrow_apply<T>(ctx, m - k, std::min(block, n - k), QR + (int64_t)k * lda + k, lda,
                              Tm + (size_t)p * kNarrow * kNarrow, 0, Q + (int64_t)k * ldq + k, ldq, n - k, (T*)nullptr, 0, 0));
    }
    return NMX_OK;
  }
  void* ws = nullptr;
  NMX_TRY(nmx_workspace(ctx, reflector_bytes<T>(m, block, n), &ws));
  const Reflector<T> w = carve<T>(ws, m, block, n);
  const int steps = ceil_div(n, block);
  for (int s = steps - 1; s >= 0; s--) {
    const int k = s * block;
    const int nb = std::min(block, n - k);
    NMX_TRY(build_reflector<T>(ctx, w, m, QR, lda, tau, k, nb));
    NMX_TRY(apply_reflector<T>(ctx, w, m - k, nb, n - k, 0, Q + (int64_t)k * ldq + k, ldq));
  }
  return NMX_OK;
}

template <typename T>
int qr_r_api(nmx_ctx* ctx, int n, const T* QR, int lda, T* R, int ldr) {
  if (!ctx) return -1;
  if (n < 0) return -2;
  if (lda < std::max(1, n)) return -4;
  if (ldr < std::max(1, n)) return -6;
  if (n == 0) return NMX_OK;
  if (!QR) return -3;
  if (!R) return -5;
  upper_kernel<T><<<(unsigned)(((int64_t)n * n + 255) / 256), 256, 0, ctx->stream>>>(n, QR, lda, R, ldr);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

template <typename T>
int gels_api(nmx_ctx* ctx, int m, int n, int nrhs, T* A, int lda, T* tau, T* B, int ldb, int block) {
  if (!ctx) return -1;
  if (m < 0) return -2;
  if (n < 1 || n > m) return -3;
  if (nrhs < 0) return -4;
  if (lda < n) return -6;
  if (ldb < std::max(1, nrhs)) return -9;
  if (block < 1 || block > kQrMaxBlock) return -10;
  if (nrhs == 0) return NMX_OK;
  if (!A) return -5;
  if (!tau) return -7;
  if (!B) return -8;
  if (block <= kNarrow) {
    NMX_TRY(geqrf_narrow<T>(ctx, m, n, A, lda, tau, block, B, ldb, nrhs));
  } else {
    NMX_TRY(geqrf_impl<T>(ctx, m, n, A, lda, tau, block));
    NMX_TRY(ormqr_impl<T>(ctx, 1, m, n, nrhs, A, lda, tau, B, ldb, block));
  }
  return trsm_left<T>(ctx, 1, 0, 0, n, nrhs, A, lda, B, ldb);
}

}  // namespace

NMX_API int nmx_geqrf_f64(nmx_ctx* ctx, int m, int n, double* A, int lda, double* tau, int block) {
  return geqrf_api<double>(ctx, m, n, A, lda, tau, block);
}
NMX_API int nmx_geqrf_f32(nmx_ctx* ctx, int m, int n, float* A, int lda, float* tau, int block) {
  return geqrf_api<float>(ctx, m, n, A, lda, tau, block);
}

NMX_API int nmx_ormqr_f64(nmx_ctx* ctx, int trans, int m, int n, int nrhs, const double* QR, int lda,
                          const double* tau, double* B, int ldb, int block) {
  return ormqr_api<double>(ctx, trans, m, n, nrhs, QR, lda, tau, B, ldb, block);
}
NMX_API int nmx_ormqr_f32(nmx_ctx* ctx, int trans, int m, int n, int nrhs, const float* QR, int lda,
                          const float* tau, float* B, int ldb, int block) {
  return ormqr_api<float>(ctx, trans, m, n, nrhs, QR, lda, tau, B, ldb, block);
}

NMX_API int nmx_orgqr_f64(nmx_ctx* ctx, int m, int n, const double* QR, int lda, const double* tau, double* Q,
                          int ldq, int block) {
  return orgqr_api<double>(ctx, m, n, QR, lda, tau, Q, ldq, block);
}
NMX_API int nmx_orgqr_f32(nmx_ctx* ctx, int m, int n, const float* QR, int lda, const float* tau, float* Q, int ldq,
                          int block) {
  return orgqr_api<float>(ctx, m, n, QR, lda, tau, Q, ldq, block);
}

NMX_API int nmx_qr_r_f64(nmx_ctx* ctx, int n, const double* QR, int lda, double* R, int ldr) {
  return qr_r_api<double>(ctx, n, QR, lda, R, ldr);
}
NMX_API int nmx_qr_r_f32(nmx_ctx* ctx, int n, const float* QR, int lda, float* R, int ldr) {
  return qr_r_api<float>(ctx, n, QR, lda, R, ldr);
}

NMX_API int nmx_gels_f64(nmx_ctx* ctx, int m, int n, int nrhs, double* A, int lda, double* tau, double* B, int ldb,
                         int block) {
  return gels_api<double>(ctx, m, n, nrhs, A, lda, tau, B, ldb, block);
}
NMX_API int nmx_gels_f32(nmx_ctx* ctx, int m, int n, int nrhs, float* A, int lda, float* tau, float* B, int ldb,
                         int block) {
  return gels_api<float>(ctx, m, n, nrhs, A, lda, tau, B, ldb, block);
}
