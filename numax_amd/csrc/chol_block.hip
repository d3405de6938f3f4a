// Cholesky of one diagonal block, up to 128 (FP64) or 256 (FP32) columns, in
// one workgroup: potrf_diag (numax/linalg/panel.mojo:216-286) and the panel
// recursion around it.  d <= 0 is floored to 1e-30 with the first failure
// recorded 1-based.
//
// Wavefront w holds block row w as 16 x 16 tiles in registers, each transposed
// in the MFMA output layout: a tile is then both operands of the update
// C_ij -= X_i X_j^T as it is, and the right operand of X = C L_ss^-T.  Step s:
// wavefront s factors its diagonal tile, a row per lane with the pivot column
// by DPP broadcast, and publishes the tile and its inverse; barrier; the
// wavefronts below form X (one correction by the residual, as accurate as
// substitution), store it and publish it; barrier; they update their tiles,
// the diagonal one first, each product written one place down so that the
// next step's column is always tile 0 and the loop over steps stays rolled.
//
// What bounds it: the chain of 16-column steps, mostly the diagonal tile's 16
// dependent columns.  Root and reciprocal of a pivot come from one
// Goldschmidt iteration on v_rsq with residual corrections, and a column's
// quotients are products corrected by their residuals; a pivot out
// of their range (negative, zero, tiny, huge, NaN) sends the tile through the
// plain square roots and divisions, and a tile of X that is not finite through
// plain substitution.  64 columns a launch with a
// barrier per column took 55 us FP64 (27 us for 32 columns FP32), and a 128
// column block two of them, a triangular solve and a product.
// 128 columns FP64: 36 us; 256 columns FP32: 75 us.  FP64 Cholesky + solve of
// order 8192: 21.2 -> 14.5 ms when this replaced the recursion, 13.4 with the
// thin products; order 1301 FP32 2.3 -> 1.2 ms.
#include "tile16.h"

namespace {

constexpr double kFloor = 1e-30;  // numax/linalg/common.mojo:27-29

// root = sqrt(d) and rinv = 1 / root of a d in the range below, the rounding of
// each left to one correction by its own residual.
__device__ __forceinline__ bool plain_pivot(double d) { return d >= 1e-280 && d <= 1e280; }
__device__ __forceinline__ bool plain_pivot(float d) { return d >= 1e-30f && d <= 1e30f; }
__device__ __forceinline__ void root_pair(double d, double& root, double& rinv) {
  const double y = __builtin_amdgcn_rsq(d);
  double g = d * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  const double t = h + h;
  g = __builtin_fma(__builtin_fma(-g, g, d), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, d), h, g);
  root = g;
  rinv = __builtin_fma(__builtin_fma(-t, g, 1.0), t, t);
}
__device__ __forceinline__ void root_pair(float d, float& root, float& rinv) {
  const float y = __builtin_amdgcn_rsqf(d);
  float g = d * y, h = 0.5f * y;
  const float r = __builtin_fmaf(-h, g, 0.5f);
  g = __builtin_fmaf(g, r, g);
  h = __builtin_fmaf(h, r, h);
  const float t = h + h;
  g = __builtin_fmaf(__builtin_fmaf(-g, g, d), h, g);
  root = g;
  rinv = __builtin_fmaf(__builtin_fmaf(-t, g, 1.f), t, t);
}

// Row I of column c of the inverse of the lower triangular block whose rows
// the 16 lanes hold (m: row `lane % 16`, rinv: the reciprocal of its diagonal);
// ny is the inverse's column negated.
template <int I, typename T>
__device__ __forceinline__ void invert_rows(const T (&m)[16], T rinv, int c, T (&ny)[16]) {
  if constexpr (I < 16) {
    T s0 = I == c ? T(1) : T(0), s1 = T(0);
#pragma unroll
    for (int j = 0; j < I; j++) fmac_bcast<I>(j & 1 ? s1 : s0, m[j], ny[j]);
    const T q = (s0 + s1) * row_bcast<I>(rinv);
    ny[I] = I < c ? T(0) : -q;
    invert_rows<I + 1, T>(m, rinv, c, ny);
  }
}

// m[C] -= l * (lane C's m[J]) for the columns right of J
template <int J, int C, typename T>
__device__ __forceinline__ void chol_update(T (&m)[16], T nl) {
  if constexpr (C < 16) {
    fmac_bcast<C>(m[C], m[J], nl);
    chol_update<J, C + 1>(m, nl);
  }
}

// Columns J .. 15 of a whole 16 x 16 tile whose row lc this lane holds (every
// 16-lane row of the wavefront holds the same).  No branches: a pivot or
// quotient out of the plain range sets `odd`, and the tile is then factored
// again by chol_tile_general.  own_rinv: 1 / this row's diagonal entry.
template <int J, typename T>
__device__ __forceinline__ void chol_columns(T (&m)[16], T& own_rinv, int lc, bool& odd) {
  if constexpr (J < 16) {
    const T d = row_bcast<J>(m[J]);
    T root, rinv;
    root_pair(d, root, rinv);
    // m / root: the product with the reciprocal, corrected by its residual
    const T q = m[J] * rinv;
    const T q2 = __builtin_elementwise_fma(__builtin_elementwise_fma(-q, root, m[J]), rinv, q);
    odd = odd || !plain_pivot(d) || q2 != q2;
    m[J] = lc > J ? q2 : root;
    own_rinv = lc == J ? rinv : own_rinv;
    chol_update<J, J + 1>(m, -m[J]);
    chol_columns<J + 1>(m, own_rinv, lc, odd);
  }
}

// potrf_diag's own arithmetic on the tile in D (cols <= 16 real columns) by
// lanes 0..15: the floor, the first failure, square roots and divisions.
template <typename T>
__device__ __forceinline__ void chol_tile_general(T (*D)[17], int lane, int cols, int col0, bool& info_set,
                                                  int32_t* info) {
#pragma unroll 1
  for (int j = 0; j < cols; j++) {
    const T d = D[j][j];
    if (d <= T(0) && !info_set) {
      info_set = true;
      if (lane == 0) *info = col0 + j + 1;
    }
    const T root = sqrt(d <= T(0) ? T(kFloor) : d);
    const T l = lane < 16 ? D[lane][j] / root : T(0);
    wave_lds_order();
    if (lane < 16 && lane >= j) D[lane][j] = lane > j ? l : root;
    wave_lds_order();
    if (lane < 16) {
#pragma unroll 1
      for (int c = j + 1; c <= lane; c++) D[lane][c] = D[lane][c] - l * D[c][j];
    }
    wave_lds_order();
  }
}

// x = c L_ss^-T by plain substitution, a row per lane 0..15, in the wavefront's
// own LDS tile: where a quotient is not finite, so that an infinity or NaN
// spreads to the columns right of it and no others, and an infinite pivot
// gives zeros.
template <typename T>
__device__ __forceinline__ void chol_substitute(const T (*D)[17], T (*tile)[64], int lane, const typename Acc<T>::type& c,
                                                typename Acc<T>::type& x) {
#pragma unroll
  for (int e = 0; e < 4; e++) tile[e][lane] = c[e];
  wave_lds_order();
  if (lane < 16) {
    auto at = [&](int j) -> T& { return sizeof(T) == 8 ? tile[j >> 2][16 * (j & 3) + lane] : tile[j & 3][16 * (j >> 2) + lane]; };
#pragma unroll 1
    for (int j = 0; j < 16; j++) {
      const T l = at(j) / D[j][j];
      at(j) = l;
#pragma unroll 1
      for (int i = j + 1; i < 16; i++) at(i) = at(i) - l * D[i][j];
    }
  }
  wave_lds_order();
#pragma unroll
  for (int e = 0; e < 4; e++) x[e] = tile[e][lane];
}

template <typename T, int NB16>
struct CholLds {
  T D[16][17];         // the step's factored diagonal tile, row-major
  T inv[16][17];       // its inverse
  T x[NB16][4][64];    // -X_w of the step, as held
  int info_set;
};

template <typename T, int NB16>
__global__ void __launch_bounds__(64 * NB16) chol_block_kernel(T* __restrict__ A, int lda, int k0, int nb,
                                                               int32_t* __restrict__ info) {
  typedef typename Acc<T>::type acc_t;
  __shared__ CholLds<T, NB16> L;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lc = lane & 15;
  const int steps = (nb + 15) / 16;
  if (t == 0) L.info_set = *info != 0;
  // held tile (w, j): lane's item e is row 16 w + lc, column 16 j + acc_row
  T* const row = A + (int64_t)(k0 + 16 * w + lc) * lda + k0;
  const bool in = 16 * w + lc < nb;
  acc_t c[NB16 - 1], dg;
#pragma unroll
  for (int j = 0; j < NB16 - 1; j++) {
    c[j] = acc_t{0, 0, 0, 0};
    if (j < w && j < steps) {  // uniform
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int col = 16 * j + acc_row<T>(lane, e);
        c[j][e] = in ? row[col] : T(0);  // columns left of the diagonal tile are all inside
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int col = acc_row<T>(lane, e);
    dg[e] = in && col <= lc ? row[16 * w + col] : T(0);
  }
  __syncthreads();
#pragma unroll 1
  for (int s = 0; s < steps; s++) {
    if (w == s) {
#pragma unroll
      for (int e = 0; e < 4; e++) L.D[lc][acc_row<T>(lane, e)] = dg[e];
      wave_lds_order();
      T m[16];
#pragma unroll
      for (int j = 0; j < 16; j++) m[j] = L.D[lc][j];
      T rinv = T(1);
      bool odd = nb - 16 * s < 16;
      chol_columns<0>(m, rinv, lc, odd);
      if (__ballot(odd)) {
        bool set = L.info_set != 0;
        chol_tile_general<T>(L.D, lane, min(16, nb - 16 * s), k0 + 16 * s, set, info);
        if (lane == 0 && set) L.info_set = 1;
#pragma unroll
        for (int j = 0; j < 16; j++) m[j] = L.D[lc][j];
        rinv = in ? T(1) / L.D[lc][lc] : T(1);  // rows past nb: the identity
      }
      T ny[16];
      invert_rows<0, T>(m, rinv, lc, ny);
      if (lane < 16) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
          L.D[lc][j] = j <= lc ? m[j] : T(0);
          L.inv[j][lc] = -ny[j];
        }
      }
    }
    __syncthreads();
    if (w > s && w < steps) {
      T iv[4], ld[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        iv[q] = L.inv[lc][acc_row<T>(lane, q)];
        ld[q] = L.D[lc][acc_row<T>(lane, q)];
      }
      acc_t x = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4; q++) x = mma(iv[q], c[0][q], x);
      acc_t res = c[0];
#pragma unroll
      for (int q = 0; q < 4; q++) res = mma(ld[q], -x[q], res);
#pragma unroll
      for (int q = 0; q < 4; q++) x = mma(iv[q], res[q], x);
      bool bad = false;
#pragma unroll
      for (int e = 0; e < 4; e++) bad = bad || !finite(x[e]);
      if (__ballot(bad)) chol_substitute<T>(L.D, L.x[w], lane, c[0], x);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        L.x[w][e][lane] = -x[e];
        if (in) row[16 * s + acc_row<T>(lane, e)] = x[e];
      }
      c[0] = x;
    } else if (w == s) {
      // the diagonal tile's lower triangle
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int col = acc_row<T>(lane, e);
        if (in && col <= lc) row[16 * w + col] = L.D[lc][col];
      }
    }
    __syncthreads();
    if (w > s && w < steps) {
      // products from zero, one addition each: summed onto the tile every term
      // would round at the tile's size (256 columns FP32: 2.4x the error)
      const acc_t x = c[0];
      acc_t d = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4; q++) d = mma(L.x[w][q][lane], x[q], d);
      dg += d;
      // tile j of the row moves to place j - 1 with the product
#pragma unroll
      for (int j = 1; j < NB16 - 1; j++)
        if (j < w - s) {  // uniform
          acc_t v = {0, 0, 0, 0};
#pragma unroll
          for (int q = 0; q < 4; q++) v = mma(L.x[s + j][q][lane], x[q], v);
          c[j - 1] = c[j] + v;
        }
    }
    // the next step's X is published after its first barrier, which every
    // wavefront reaches only after its reads here
  }
}

}  // namespace

template <typename T>
int chol_block(nmx_ctx* ctx, T* A, int lda, int k0, int nb, int32_t* info) {
  constexpr int kMax16 = chol_block_max<T>() / 16;
  if (nb > 16 * kMax16) return NMX_ERR_UNSUPPORTED;
  ProfScope ps(ctx, K_POTRF_DIAG, (double)nb * nb * nb / 3.0, 2.0 * sizeof(T) * nb * nb);
  // the smaller workgroup while it holds the block: its barriers are shorter
  if (nb <= 64) chol_block_kernel<T, 4><<<1, 64 * 4, 0, ctx->stream>>>(A, lda, k0, nb, info);
  else if (nb <= 128) chol_block_kernel<T, 8><<<1, 64 * 8, 0, ctx->stream>>>(A, lda, k0, nb, info);
  else chol_block_kernel<T, kMax16><<<1, 64 * kMax16, 0, ctx->stream>>>(A, lda, k0, nb, info);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}
template int chol_block<double>(nmx_ctx*, double*, int, int, int, int32_t*);
template int chol_block<float>(nmx_ctx*, float*, int, int, int, int32_t*);
