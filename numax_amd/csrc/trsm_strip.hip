// Triangular solve with a triangle of at most 256 rows, op(T) X = B in place,
// one launch: the base of the recursive TRSM (trsm_diag / _trsm,
// numax/linalg/panel.mojo:2221-2276, triangular.mojo:114-225) for every
// triangle, transposition and vector layout.
//
// A workgroup of four wavefronts takes 16 or 32 vectors through the whole
// triangle in 16-row blocks.  In solve order op(T) is lower triangular (an
// upper one is read from its last row up), block s of it belongs to wavefront
// s % 4, and a block's right-hand sides stay in the owner's registers in the
// MFMA output layout.  Step s: the owner multiplies its block by the inverse
// of the 16 x 16 diagonal block, corrects that by its residual, and passes
// X_s on through LDS; one barrier; every wavefront subtracts its blocks'
// products with X_s.  The products run
// on 16x16x4 MFMA with the contraction index permuted to the output layout's
// row order, so an output is the next product's operand as it is.  The tiles
// of T do not depend on X and are read a step ahead.
//
// What bounds it: the chain of 16-row steps (four products of one tile, an LDS
// round and a barrier each).  64 rows a launch by substitution, a column per
// thread, took 15 us (FP64 or FP32, 64 rows) and a GEMM launch between every
// two: 256 rows by 7936 columns FP64 were 4 such launches and 3 GEMMs.
// Now 256 rows by 16 columns FP64 are one launch of 23 us, 64 rows 6 us: FP64
// Cholesky + 16-column solve of order 8192 31.7 -> 21.2 ms (11.8 with the
// Cholesky blocks and thin products since).
//
// The inverses are of 16 x 16 blocks only and made per workgroup (a column
// per lane, the block's rows by DPP broadcast).  A workgroup that meets a
// non-finite inverse or solution solves its vectors again by plain
// substitution, so that an infinity or NaN spreads as far as substitution
// spreads it and no further.
#include "tile16.h"

namespace {

struct StripArgs {
  int n, nvec;
  int sr, sk;       // element (r, k) of op(T) at r sr + k sk
  int upper, unit;
  int br;           // B's entry of row r and vector v at r br + v bv
  int64_t bv;
};

constexpr int kStripThreads = 256;

template <typename T, int NS, int NV>
struct StripLds {
  T x[2][NV][4][64];      // -X_s in the output layout, by step parity
  T inv[4 * NS][16][17];  // diagonal blocks' inverses
  int bad;
};

// One step's tiles of T for this wavefront's blocks, block 4 u + w against
// block S.  Called only while a block follows S, so that S is whole and the
// column offset (koff + S kstep) is inside the triangle; a row past n has an
// offset that no such addend brings back into the descriptor's range.
template <int S, typename T, int NS>
__device__ __forceinline__ void strip_tiles(__amdgpu_buffer_rsrc_t rt, const uint32_t (&rowoff)[NS],
                                            const uint32_t (&koff)[4], uint32_t kstep, int w, T (&tl)[NS][4]) {
#pragma unroll
  for (int u = S >> 2; u < NS; u++) {
    if (u > S >> 2 || w > (S & 3)) {  // uniform
#pragma unroll
      for (int q = 0; q < 4; q++) tl[u][q] = buf_load<T>(rt, rowoff[u] + (koff[q] + (uint32_t)S * kstep));
    }
  }
}

template <int S, typename T, int NS, int NV>
__device__ __forceinline__ void strip_steps(int n, __amdgpu_buffer_rsrc_t rt, const uint32_t (&rowoff)[NS],
                                            const uint32_t (&koff)[4], uint32_t kstep, int w, int lane,
                                            typename Acc<T>::type (&r)[NS][NV], const T (&iv)[NS][4],
                                            const T (&dg)[NS][4], bool& bad,
                                            T (&tl)[2][NS][4], StripLds<T, NS, NV>& L) {
  if constexpr (S < 4 * NS) {
    constexpr int u = S >> 2, owner = S & 3, buf = S & 1;
    if (16 * S < n) {  // uniform
      // the next step's tiles are issued here and not earlier (they depend on
      // nothing, and all steps' tiles at once do not fit the registers)
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (S + 2 < 4 * NS)
        if (16 * (S + 2) < n) strip_tiles<S + 1, T, NS>(rt, rowoff, koff, kstep, w, tl[buf ^ 1]);
      if (w == owner) {
#pragma unroll
        for (int g = 0; g < NV; g++) {
          typename Acc<T>::type x = {0, 0, 0, 0};
          // x = inv r, then one correction by the block's own residual: with
          // it the step is as accurate as substitution (without it a factor
          // with small pivots, unpivoted LU, failed to converge in refinement)
#pragma unroll
          for (int q = 0; q < 4; q++) x = mma(iv[u][q], r[u][g][q], x);
          typename Acc<T>::type res = r[u][g];
#pragma unroll
          for (int q = 0; q < 4; q++) res = mma(dg[u][q], -x[q], res);
#pragma unroll
          for (int q = 0; q < 4; q++) x = mma(iv[u][q], res[q], x);
          r[u][g] = x;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            bad = bad || !finite(x[e]);
            L.x[buf][g][e][lane] = -x[e];
          }
        }
      }
      if (16 * (S + 1) < n) {  // uniform: a later block waits for X_S
        // two buffers: X_S+2 is written after the barrier of step S + 1, which
        // each wavefront reaches only after its reads of X_S
        __syncthreads();
#pragma unroll
        for (int g = 0; g < NV; g++) {
          T xb[4];
#pragma unroll
          for (int q = 0; q < 4; q++) xb[q] = L.x[buf][g][q][lane];
#pragma unroll
          for (int v = u; v < NS; v++)
            if (v > u || w > owner) {  // uniform
              // the product from zero, then one addition: summed onto r each
              // of its terms would round at r's size (256 rows: 1.8x the error)
              typename Acc<T>::type d = {0, 0, 0, 0};
#pragma unroll
              for (int q = 0; q < 4; q++) d = mma(tl[buf][v][q], xb[q], d);
              r[v][g] += d;
            }
        }
      }
    }
    strip_steps<S + 1, T, NS, NV>(n, rt, rowoff, koff, kstep, w, lane, r, iv, dg, bad, tl, L);
  }
}

template <typename T, int NS, int NV>
__global__ void __launch_bounds__(kStripThreads) __attribute__((amdgpu_waves_per_eu(2)))
trsm_strip_kernel(StripArgs a, const T* __restrict__ Tm, T* __restrict__ B) {
  __shared__ StripLds<T, NS, NV> L;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lc = lane & 15, lk = lane >> 4;
  const int n = a.n, v0 = blockIdx.x * 16 * NV;
  constexpr uint32_t E = sizeof(T);
  constexpr uint32_t kOut = 0x80000000u;  // stays out of range under any in-range addend
  const __amdgpu_buffer_rsrc_t rt = buf_rsrc(Tm);
  const __amdgpu_buffer_rsrc_t rb = buf_rsrc(B + v0 * a.bv);
  if (t == 0) L.bad = 0;
  // the diagonal block this lane inverts a column of: block 4 lk + w, its row lc here
  T m[16];
  const int d0 = 16 * (4 * lk + w), dr = d0 + lc, pr = a.upper ? n - 1 - dr : dr;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const int pk = a.upper ? n - 1 - (d0 + j) : d0 + j;
    const uint32_t off = ((uint32_t)pr * (uint32_t)a.sr + (uint32_t)pk * (uint32_t)a.sk) * E;
    const bool in = dr < n && (a.unit ? j < lc : j <= lc);
    m[j] = buf_load<T>(rt, in ? off : kBufOob);
  }
  uint32_t rowoff[NS], koff[4];
#pragma unroll
  for (int u = 0; u < NS; u++) {
    const int row = 16 * (4 * u + w) + lc;
    rowoff[u] = row < n ? (uint32_t)(a.upper ? n - 1 - row : row) * (uint32_t)a.sr * E : kOut;
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int k = acc_row<T>(lane, q);
    koff[q] = (uint32_t)(a.upper ? n - 1 - k : k) * (uint32_t)a.sk * E;
  }
  const uint32_t kstep = (uint32_t)(a.upper ? -16 : 16) * (uint32_t)a.sk * E;
  T tl[2][NS][4];
  if (n > 16) strip_tiles<0, T, NS>(rt, rowoff, koff, kstep, w, tl[0]);
  typename Acc<T>::type r[NS][NV];
  auto boff = [&](int u, int g, int e) {
    const int row = 16 * (4 * u + w) + acc_row<T>(lane, e), v = 16 * g + lc;
    const int p = a.upper ? n - 1 - row : row;
    return row < n && v0 + v < a.nvec ? ((uint32_t)p * (uint32_t)a.br + (uint32_t)v * (uint32_t)a.bv) * E : kBufOob;
  };
#pragma unroll
  for (int u = 0; u < NS; u++)
#pragma unroll
    for (int g = 0; g < NV; g++)
#pragma unroll
      for (int e = 0; e < 4; e++) r[u][g][e] = buf_load<T>(rb, boff(u, g, e));
  // the diagonal blocks themselves, as MFMA operands
  T dg[NS][4];
#pragma unroll
  for (int u = 0; u < NS; u++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int k = acc_row<T>(lane, q), row = 16 * (4 * u + w) + lc, col = 16 * (4 * u + w) + k;
      const uint32_t off = rowoff[u] + (uint32_t)(a.upper ? n - 1 - col : col) * (uint32_t)a.sk * E;
      const bool in = row < n && (a.unit ? k < lc : k <= lc);
      const T v = buf_load<T>(rt, in ? off : kBufOob);
      dg[u][q] = a.unit && k == lc ? T(1) : v;
    }
  T diag = T(1);
#pragma unroll
  for (int j = 0; j < 16; j++)
    if (j == lc && dr < n && !a.unit) diag = m[j];
  const T rinv = T(1) / diag;
  T ny[16];
  invert_rows<0, T>(m, rinv, lc, ny);
  bool bad = false;
  if (lk < NS) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      bad = bad || !finite(ny[i]);
      L.inv[4 * lk + w][i][lc] = -ny[i];
    }
  }
  wave_lds_order();
  T iv[NS][4];
#pragma unroll
  for (int u = 0; u < NS; u++)
#pragma unroll
    for (int q = 0; q < 4; q++) iv[u][q] = L.inv[4 * u + w][lc][acc_row<T>(lane, q)];
  strip_steps<0, T, NS, NV>(n, rt, rowoff, koff, kstep, w, lane, r, iv, dg, bad, tl, L);
  if (bad) L.bad = 1;
  __syncthreads();
  if (L.bad) {
    // plain substitution in place, a vector per thread
    if (t < 16 * NV && v0 + t < a.nvec) {
      T* b = B + (int64_t)(v0 + t) * a.bv;
#pragma unroll 1
      for (int j = 0; j < n; j++) {
        const int pj = a.upper ? n - 1 - j : j;
        const T* col = Tm + (int64_t)pj * a.sk;
        const T xj = a.unit ? b[(int64_t)pj * a.br] : b[(int64_t)pj * a.br] / col[(int64_t)pj * a.sr];
        b[(int64_t)pj * a.br] = xj;
#pragma unroll 1
        for (int i = j + 1; i < n; i++) {
          const int pi = a.upper ? n - 1 - i : i;
          b[(int64_t)pi * a.br] -= col[(int64_t)pi * a.sr] * xj;
        }
      }
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < NS; u++)
#pragma unroll
    for (int g = 0; g < NV; g++)
#pragma unroll
      for (int e = 0; e < 4; e++) buf_store(rb, boff(u, g, e), r[u][g][e]);
}

template <typename T, int NS>
void strip_run(nmx_ctx* ctx, const StripArgs& a, const T* Tm, T* B) {
  // 16 vectors a workgroup while there is a CU for each workgroup; above that
  // 32, which halve the reads of T (and 256 rows of 16 take all of a CU's
  // registers, so a second round of workgroups would wait for the first)
  if (a.nvec > 16 * ctx->num_cus)
    trsm_strip_kernel<T, NS, 2><<<ceil_div(a.nvec, 32), kStripThreads, 0, ctx->stream>>>(a, Tm, B);
  else
    trsm_strip_kernel<T, NS, 1><<<ceil_div(a.nvec, 16), kStripThreads, 0, ctx->stream>>>(a, Tm, B);
}

}  // namespace

template <typename T>
int trsm_strip(nmx_ctx* ctx, int upper, int unit, int trans, int vec_rows, int n, int nvec, const T* Tm, int ldt, T* B,
               int ldb) {
  if (n > kStripMax) return NMX_ERR_UNSUPPORTED;
  const StripArgs a{n, nvec, trans ? 1 : ldt, trans ? ldt : 1, upper, unit, vec_rows ? 1 : ldb, vec_rows ? ldb : 1};
  ProfScope ps(ctx, K_TRSM, (double)n * n * nvec, sizeof(T) * ((double)n * n + 2.0 * n * nvec));
  if (n <= 64) strip_run<T, 1>(ctx, a, Tm, B);
  else if (n <= 128) strip_run<T, 2>(ctx, a, Tm, B);
  else strip_run<T, 4>(ctx, a, Tm, B);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}
template int trsm_strip<double>(nmx_ctx*, int, int, int, int, int, int, const double*, int, double*, int);
template int trsm_strip<float>(nmx_ctx*, int, int, int, int, int, int, const float*, int, float*, int);
