// Triangular solve with a triangle of at most 256 rows, op(T) X = B in place,
// one launch: the base of the recursive TRSM (trsm_diag / _trsm,
// numax/linalg/panel.mojo:2221-2276, triangular.mojo:114-225) for every
// triangle, transposition and vector layout.
//
// The order of every sum is that of substitution in blocks of 64 rows, split
// in two at multiples of 64 the way trsm_rec splits above 256: inside a block
// a row subtracts one product after another, each rounded once, and takes a
// correctly rounded quotient; between blocks a product over all rows of the
// half solved before is summed from zero in ascending order of the stored
// index and subtracted once.  Results do not depend on where a strip ends.
// (MFMA of FP64 and FP32 is a chain of fused multiply-adds over its four
// contraction indices in ascending order, measured over random operands down
// to the subnormals, so a product taken four rows at a time keeps the order.)
//
// A workgroup of four wavefronts takes 16 or 32 vectors through the whole
// triangle in 16-row steps; wavefront w owns rows 16 w .. 16 w + 15 of each
// 64-row block and holds their right-hand sides in the MFMA output layout.
// In solve order op(T) is lower triangular (an upper one is read from its
// last row up, padded at that end to whole blocks).  A step: the owner puts its tile in LDS, reads
// it back a vector per lane, substitutes (the diagonal tile's rows reach the
// lanes as the DPP operand of the multiply-adds), and passes X on through LDS;
// one barrier; the block's later wavefronts subtract their products with it.
// After a block's last step come the products onto later blocks.
//
// What bounds it: the chain of 16-row steps (120 multiply-adds, an LDS round
// and a barrier each, 0.9 us; 1.2 with quotients) and the reads of a
// row-major triangle, 16 rows to an instruction.  A quotient is the product
// with the diagonal's reciprocal and two corrections by its residual; a tile
// that meets an operand outside their range is solved again with divisions.
// 16 vectors, FP64, unit / non-unit: 64 rows 7.4 / 9.4 us, 256 rows 28.7 / 34.6.
// A launch a 64-row block with a column per thread and products between took
// 16 / 19 and 87 / 100 us for the same bits.  Multiplied by inverses of the
// 16 x 16 diagonal tiles with one correction, 256 rows took 24 us, but in
// LU solves of Gaussian systems of order 8192 that order of operations had
// 1.6 times the error (geometric mean over 16 systems against a refined solution).
#include "tile16.h"

namespace {

struct StripArgs {
  int n, npad, nvec;  // npad: n rounded up to whole 64-row blocks
  int sr, sk;         // element (r, k) of op(T) at r sr + k sk
  int upper;
  int halves;         // three blocks that split 1 + 2 in solve order instead of 2 + 1
  int br;             // B's entry of row r and vector v at r br + v bv
  int64_t bv;
};

constexpr int kStripThreads = 256;

// x[I] += (lane I's m) * y for the rows I .. 15
template <int I, typename T>
__device__ __forceinline__ void subtract_rows(T (&x)[16], T m, T y) {
  if constexpr (I + 3 < 16) {
    fmac_lanes4<I>(x[I], x[I + 1], x[I + 2], x[I + 3], m, y);
    subtract_rows<I + 4>(x, m, y);
  } else if constexpr (I < 16) {
    fmac_bcast<I>(x[I], m, y);
    subtract_rows<I + 1>(x, m, y);
  }
}

// Substitution in a 16 x 16 lower triangle whose row lane % 16 is m (strictly
// below the diagonal) and dg, for this lane's vector x.  PLAIN: divisions.
template <int J, typename T, bool UNIT, bool PLAIN>
__device__ __forceinline__ void substitute(const T (&m)[16], T dg, T rinv, T (&x)[16], int& least, int& most) {
  if constexpr (J < 16) {
    if constexpr (!UNIT) {
      const T d = row_bcast<J>(dg);
      if constexpr (PLAIN) {
        x[J] = x[J] / d;
      } else {
        least = min(least, magnitude(x[J]));
        most = max(most, magnitude(x[J]));
        x[J] = quotient(x[J], d, row_bcast<J>(rinv));
      }
    }
    if constexpr (J < 15) subtract_rows<J + 1>(x, m[J], -x[J]);
    substitute<J + 1, T, UNIT, PLAIN>(m, dg, rinv, x, least, most);
  }
}

// d[y] += (target y's tile row) (source block's solution), rows 4 Q .. of it on
template <int Q, typename T, int NS, int NV, int TARGETS>
__device__ __forceinline__ void strip_products(const T (&tg)[2][16], const T* x, int step,
                                               typename Acc<T>::type (&d)[2][NV]) {
  if constexpr (Q < 16) {
#pragma unroll
    for (int g = 0; g < NV; g++) {
      const T xq = x[g * (64 * NS * 16) + Q * step];
      d[0][g] = mma(tg[0][Q], xq, d[0][g]);
      if constexpr (TARGETS == 2) d[1][g] = mma(tg[1][Q], xq, d[1][g]);
    }
    strip_products<Q + 1, T, NS, NV, TARGETS>(tg, x, step, d);
  }
}

template <typename T, int NS, int NV, bool UNIT>
__global__ void __launch_bounds__(kStripThreads) __attribute__((amdgpu_waves_per_eu(2)))
trsm_strip_kernel(StripArgs a, const T* __restrict__ Tm, T* __restrict__ B) {
  typedef typename Acc<T>::type acc_t;
  __shared__ T X[NV][64 * NS][16];  // the solution by row in solve order; a step's right-hand sides before it
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lc = lane & 15, lk = lane >> 4;
  const int n = a.n, v0 = blockIdx.x * 16 * NV;
  constexpr uint32_t E = sizeof(T);
  const __amdgpu_buffer_rsrc_t rt = buf_rsrc(Tm);
  const __amdgpu_buffer_rsrc_t rb = buf_rsrc(B + v0 * a.bv);
  // stored index of row i in solve order; n or above: padding
  const int flip = a.upper ? -1 : 0, shift = a.upper ? a.npad : 0;
  auto stored = [&](int i) { return (i ^ flip) + shift; };
  // Offsets are a lane's part plus a uniform part.  A part of a row or column
  // past the edge is so large that no part of the other kind brings the sum
  // back into the descriptor's range.
  constexpr uint32_t kLaneOut = 0x80000000u, kRowOut = 0x7FFFFFFFu;
  auto lane_row = [&](int p) { return p < n ? (uint32_t)p * (uint32_t)a.sr * E : kLaneOut; };
  auto col = [&](int p) { return p < n ? (uint32_t)p * (uint32_t)a.sk * E : kRowOut; };  // p uniform
  auto lane_vec = [&](int v) { return v0 + v < a.nvec ? (uint32_t)v * (uint32_t)a.bv * E : kLaneOut; };
  const int nb = a.npad / 64;
  // 16-row steps that are padding throughout come first in an upper triangle, last in a lower one
  const int s_begin = a.upper ? (a.npad - n) / 16 : 0, s_end = a.upper ? 4 * nb : (n + 15) / 16;
  for (int i = t; i < 16 * s_begin * 16 * NV; i += kStripThreads) X[i / (16 * 16 * s_begin)][i / 16 % (16 * s_begin)][i % 16] = T(0);

  acc_t r[NS][NV];  // of this wavefront's tiles, the current block's first
#pragma unroll
  for (int u = 0; u < NS; u++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int p = stored(64 * u + 16 * w + acc_row<T>(lane, e));
      const bool in = 64 * u < a.npad && p < n;
#pragma unroll
      for (int g = 0; g < NV; g++)
        r[u][g][e] = buf_load<T>(rb, in ? lane_vec(16 * g + lc) + (uint32_t)p * (uint32_t)a.br * E : kBufOob);
    }
  // this wavefront's diagonal tile in block c, a row per lane (of what is right
  // of the diagonal nothing is used)
  T m[16], dg = T(1), rinv = T(1);
  auto load_diag = [&](int c) {
    const int i0 = 64 * c + 16 * w, pr = stored(i0 + lc);
    const uint32_t row = lane_row(pr);
#pragma unroll
    for (int j = 0; j < 15; j++) m[j] = buf_load<T>(rt, row + col(stored(i0 + j)));
    m[15] = T(0);
    if constexpr (!UNIT) {
      dg = buf_load<T>(rt, pr < n ? row + (uint32_t)pr * (uint32_t)a.sk * E : kBufOob);
      dg = pr < n ? dg : T(1);
    }
  };
  // this wavefront's tile in the columns of step s of the same block
  T tl[4];
  auto load_left = [&](int s) {
    const uint32_t row = lane_row(stored(64 * (s >> 2) + 16 * w + lc));
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int p = stored(16 * s + 4 * q + lk);
      tl[q] = buf_load<T>(rt, p < n ? row + (uint32_t)p * (uint32_t)a.sk * E : kBufOob);
    }
  };
  // a wavefront whose step in the first block is padding starts in the second
  load_diag(w < s_begin && nb > 1 ? 1 : 0);
  if (w > s_begin) load_left(s_begin);
  if (!UNIT && w == s_begin) rinv = T(1) / dg;
  [[maybe_unused]] T tg[2][16];
#pragma unroll 1
  for (int s = s_begin; s < s_end; s++) {
    const int c = s >> 2, owner = s & 3;
    // products onto later blocks follow a block's last step: onto the next
    // block, or the next two, of one solved block or two
    const bool more = NS > 1 && owner == 3 && c + 1 < nb;
    const bool two_targets = NS > 2 && (c == 0 ? a.halves != 0 : c == 1 && nb == 4);
    const bool two_sources = NS > 2 && c == 1 && !a.halves;
    // the tiles of the targets' rows in a source block's columns
    auto load_products = [&](int src) {
      const int p0 = (a.upper ? a.npad - 64 * (src + 1) : 64 * src) + lk;
      auto target = [&](T(&to)[16], int block) {
        const uint32_t off = lane_row(stored(64 * block + 16 * w + lc)) + (uint32_t)p0 * (uint32_t)a.sk * E;
#pragma unroll
        for (int q = 0; q < 16; q++) to[q] = buf_load<T>(rt, p0 + 4 * q < n ? off + 4 * q * (uint32_t)a.sk * E : kBufOob);
      };
      target(tg[0], c + 1);
      if (two_targets) target(tg[1], c + 2);
    };
    const int src0 = two_sources && !a.upper ? c - 1 : c;
    if constexpr (NS > 1) {
      // while the wavefront waits for another's step
      if (c + 1 < nb && (w == 3 ? owner == 2 || (owner == 3 && s == s_begin) : owner == 3)) load_products(src0);
    }
    if (!UNIT && w == ((owner + 1) & 3)) rinv = T(1) / dg;  // ahead of its step
    T(*const xv)[16] = &X[NV == 2 ? lk & 1 : 0][16 * s];
    if (w == owner) {
#pragma unroll
      for (int g = 0; g < NV; g++)
#pragma unroll
        for (int e = 0; e < 4; e++) X[g][16 * s + acc_row<T>(lane, e)][lc] = r[0][g][e];
      wave_lds_order();
      T x[16];
#pragma unroll
      for (int j = 0; j < 16; j++) x[j] = xv[j][lc];
      int least = 0, most = 0;
      substitute<0, T, UNIT, false>(m, dg, rinv, x, least, most);
      if constexpr (!UNIT) {
        if (__ballot(!plain_divisor(dg) || least < -plain_magnitude<T>() || most > plain_magnitude<T>())) {
#pragma unroll
          for (int j = 0; j < 16; j++) x[j] = xv[j][lc];
          substitute<0, T, UNIT, true>(m, dg, rinv, x, least, most);
        }
      }
      if (lk < NV) {
#pragma unroll
        for (int j = 0; j < 16; j++) xv[j][lc] = x[j];
      }
    }
    __syncthreads();
    if (w == owner) {
      const uint32_t vec = lk < NV ? lane_vec(16 * lk + lc) : kLaneOut;
#pragma unroll
      for (int j = 0; j < 16; j++) {
        const int p = stored(16 * s + j);  // uniform
        buf_store(rb, vec + (p < n ? (uint32_t)p * (uint32_t)a.br * E : kRowOut), xv[j][lc]);
      }
      if (c + 1 < nb) load_diag(c + 1);
    }
    if (s + 1 == s_end) break;
    if (owner < 3 && w > owner) {
#pragma unroll
      for (int g = 0; g < NV; g++)
#pragma unroll
        for (int q = 0; q < 4; q++) r[0][g] = mma(tl[q], -X[g][16 * s + 4 * q + lk][lc], r[0][g]);
    }
    if (w > ((s + 1) & 3)) load_left(s + 1);
    if constexpr (NS > 1) {
      if (more) {
        acc_t d[2][NV];
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
          for (int g = 0; g < NV; g++) d[y][g] = acc_t{0, 0, 0, 0};
        auto products = [&](int src) {
          // row lk of the source block in stored order; four rows on are `step` away
          const T* x = X[0][64 * src + (a.upper ? 63 - lk : lk)] + lc;
          const int step = a.upper ? -4 * 16 : 4 * 16;
          if (two_targets) strip_products<0, T, NS, NV, 2>(tg, x, step, d);
          else strip_products<0, T, NS, NV, 1>(tg, x, step, d);
        };
        products(src0);
        if (two_sources) {
          const int src1 = a.upper ? c - 1 : c;
          load_products(src1);
          products(src1);
        }
#pragma unroll
        for (int g = 0; g < NV; g++) {
          r[1][g] -= d[0][g];
          if constexpr (NS > 2)
            if (two_targets) r[2][g] -= d[1][g];
#pragma unroll
          for (int u = 0; u + 1 < NS; u++) r[u][g] = r[u + 1][g];
        }
      }
    }
  }
}

template <typename T, int NS, bool UNIT>
void strip_run(nmx_ctx* ctx, const StripArgs& a, const T* Tm, T* B) {
  // 16 vectors a workgroup while there is a CU for each workgroup; above that
  // 32, which halve the reads of T
  if (a.nvec > 16 * ctx->num_cus)
    trsm_strip_kernel<T, NS, 2, UNIT><<<ceil_div(a.nvec, 32), kStripThreads, 0, ctx->stream>>>(a, Tm, B);
  else
    trsm_strip_kernel<T, NS, 1, UNIT><<<ceil_div(a.nvec, 16), kStripThreads, 0, ctx->stream>>>(a, Tm, B);
}

template <typename T, bool UNIT>
void strip_any(nmx_ctx* ctx, const StripArgs& a, const T* Tm, T* B) {
  if (a.n <= 64) strip_run<T, 1, UNIT>(ctx, a, Tm, B);
  else if (a.n <= 128) strip_run<T, 2, UNIT>(ctx, a, Tm, B);
  else strip_run<T, 4, UNIT>(ctx, a, Tm, B);
}

}  // namespace

template <typename T>
int trsm_strip(nmx_ctx* ctx, int upper, int unit, int trans, int vec_rows, int n, int nvec, const T* Tm, int ldt, T* B,
               int ldb) {
  if (n > kStripMax) return NMX_ERR_UNSUPPORTED;
  const int npad = ceil_div(n, 64) * 64;
  // trsm_split puts the first half's blocks at the stored top: 128 of 130 .. 192
  // rows, 64 of 129
  const int top = trsm_split(n) / 64;
  const int halves = npad == 192 && (upper ? 3 - top : top) == 1;
  const StripArgs a{n, npad, nvec, trans ? 1 : ldt, trans ? ldt : 1, upper, halves, vec_rows ? 1 : ldb, vec_rows ? ldb : 1};
  ProfScope ps(ctx, K_TRSM, (double)n * n * nvec, sizeof(T) * ((double)n * n + 2.0 * n * nvec));
  if (unit) strip_any<T, true>(ctx, a, Tm, B);
  else strip_any<T, false>(ctx, a, Tm, B);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}
template int trsm_strip<double>(nmx_ctx*, int, int, int, int, int, int, const double*, int, double*, int);
template int trsm_strip<float>(nmx_ctx*, int, int, int, int, int, int, const float*, int, float*, int);
