// Batched tall-skinny least squares, FP32: `count` independent problems
// min ||A x - b||, A m x n row-major (n <= 32, m >= n), one workgroup each.
//
// numax's `lstsq` (numax/linalg/qr.mojo:746-821) is blocked Householder QR
// (geqr2_panel, panel.mojo:1975-2073), Q^T b applied panel by panel
// (qr.mojo:470-534), then the upper-triangular solve with R
// (qr.mojo:536-612).  Here the n reflectors are applied one column at a time
// to [A | b] held whole in registers, and x comes from R and the first n
// entries of Q^T b.
//
// What bounds it: not HBM (each problem is read once) but the chain of n
// dependent reflectors per problem -- a sum over all rows, a square root and
// a division, an update -- so the layout is chosen for the shortest step and
// two problems share a CU to fill each other's waits.
//
// Layout: a thread holds 32 rows of columns c and c + 16, c = lane % 16; the
// four 16-lane rows of a wavefront and the wavefronts hold different rows.
// The reflector's column x then reaches the other columns of its rows as a
// DPP row broadcast inside the multiply-adds, dot products need no reduction
// across columns, and what is left of the cross-lane work is one value per
// column over the row groups (two lane-swap steps in a wavefront, one LDS
// round and one barrier across them).  With a row per lane instead, every
// step reduced 33 values over 256 threads and read them back: 165 LDS reads
// and 126 shuffles a step, and 4096 problems of 1024 x 32 took 6.55 ms.
// In this layout they take 0.65 ms (10.4x; 850 GB/s of the 4.8 TB/s a copy
// reaches): the broadcasts are the DPP operand of the multiply-adds (0.64 ms
// as separate moves), 60 % of the time is issue, the rest the step's barrier
// and LDS round.
#include <math.h>

#include "tile16.h"

namespace {

constexpr int kRows = 32;              // rows a thread holds
constexpr int kGroupPad = kRows + 4;   // LDS stride of a row group's column (b128 aligned, banks apart)

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// v(lane) + v(lane ^ 16), then the same over lane ^ 32
__device__ __forceinline__ float sum_rows16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// lanes 0..31: a(lane) + a(lane + 32); lanes 32..63: b(lane - 32) + b(lane)
__device__ __forceinline__ float sum_halves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int NW>
struct GelsLds {
  float x[NW][4][kGroupPad];                               // the reflector's column, per row group
  __attribute__((aligned(16))) float part[2][NW][16][2];   // column sums by wavefront (columns c, c + 16)
  __attribute__((aligned(16))) float part_b[2][NW < 4 ? 4 : NW];
  float row[2][34];                                        // row K: columns (c, c + 16) interleaved, then b
  float R[32][33];                                         // written and read by wavefront 0 only
  float y[32];
};

// Reflector K.  Rows 0 .. K have left the registers (they are zero there; the
// finished ones' R is in LDS), so sums over all rows are sums below the diagonal:
// sigma = x^T x, beta = -sign(alpha) sqrt(alpha^2 + sigma), v = [1; x / (alpha -
// beta)], tau = (beta - alpha) / beta, and a column that is zero below its
// diagonal stays as it is (geqr2_panel's dlarfg convention).
template <int K, int NW, int SETS>
__device__ __forceinline__ void gels_step(float (&a)[SETS][kRows], float (&b)[2], int t, GelsLds<NW>& L) {
  constexpr int set = K >> 4, lk = K & 15;
  constexpr int s0 = set;  // sets before it hold finished columns only
  constexpr int buf = K & 1;
  // opaque per step: the lane masks built from t are made where they are
  // used, not hoisted (32 steps of them spilled)
  asm volatile("" : "+v"(t));
  const int lane = t & 63, wave = NW == 1 ? 0 : t >> 6;
  const int c = lane & 15, g = lane >> 4;
  if (t < 16) {
#pragma unroll
    for (int s = s0; s < SETS; s++) {
      L.row[buf][2 * c + s] = a[s][K];
      a[s][K] = 0.f;
    }
  }
  if (t == K / 2) {
    L.row[buf][32] = b[K & 1];
    b[K & 1] = 0.f;
  }
  // b is held two rows a lane: it meets the column through LDS (own wavefront, in order)
  float* xg = L.x[wave][g];
  if (c == lk) {
#pragma unroll
    for (int r = 0; r < kRows; r += 4)
      *(float4*)(xg + r) = make_float4(a[set][r], a[set][r + 1], a[set][r + 2], a[set][r + 3]);
  }
  wave_lds_order();
  const float2 xb = *(const float2*)(xg + 2 * c);
  float p[SETS];
#pragma unroll
  for (int s = s0; s < SETS; s++) {
    float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
#pragma unroll
    for (int r = 0; r < kRows; r += 4)
      fmac_bcast4<lk>(q0, q1, q2, q3, a[set][r], a[set][r + 1], a[set][r + 2], a[set][r + 3], a[s][r], a[s][r + 1],
                      a[s][r + 2], a[s][r + 3]);
    p[s] = (q0 + q1) + (q2 + q3);
  }
  float pb = xb.x * b[0] + xb.y * b[1];
  pb = dpp_add<0xB1>(pb);   // quad_perm 1,0,3,2
  pb = dpp_add<0x4E>(pb);   // quad_perm 2,3,0,1
  pb = dpp_add<0x141>(pb);  // row_half_mirror
  pb = dpp_add<0x140>(pb);  // row_mirror
  if constexpr (SETS - s0 == 2) {
    const float v = sum_rows16(sum_halves(p[0], p[1]));
    if (g == 0 || g == 2) L.part[buf][wave][c][g >> 1] = v;
  } else {
    const float v = sum_rows16(sum_halves(p[SETS - 1], p[SETS - 1]));
    if (g == 0) L.part[buf][wave][c][SETS - 1] = v;
  }
  pb = sum_rows16(sum_halves(pb, pb));
  if (lane == 0) L.part_b[buf][wave] = pb;
  if (NW == 1) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
  float tot[2] = {0.f, 0.f}, tb = 0.f;
#pragma unroll(NW < 4 ? NW : 4)
  for (int w = 0; w < NW; w++) {
    const float2 v = *(const float2*)L.part[buf][w][c];
    tot[0] += v.x;
    tot[1] += v.y;
    tb += L.part_b[buf][w];
  }
  const float2 rk = *(const float2*)&L.row[buf][2 * c];
  const float bk = L.row[buf][32];
  const float sigma = row_bcast<lk>(tot[set]);
  const float alpha = row_bcast<lk>(set ? rk.y : rk.x);
  const bool none = sigma == 0.f;
  const float beta = none ? alpha : -copysignf(sqrtf(fmaf(alpha, alpha, sigma)), alpha);
  const float tau = (beta - alpha) / beta, scale = 1.f / (alpha - beta);
  float f[SETS];
#pragma unroll
  for (int s = s0; s < SETS; s++) {
    const float rks = s ? rk.y : rk.x;
    // finished columns, K itself and every column of a reflector that is none stay
    const float fs = 16 * s + c > K && !none ? tau * (rks + scale * tot[s]) : 0.f;
    if (t < 16) {
      const int col = 16 * s + c;
      if (col >= K) L.R[K][col] = col == K ? beta : rks - fs;
    }
    f[s] = none ? 0.f : fs * scale;
  }
  const float fy = none ? 0.f : tau * (bk + scale * tb), fb = none ? 0.f : fy * scale;
  if (t == 0) L.y[K] = bk - fy;
  // the other sets first: x is read from its own set's registers
#pragma unroll
  for (int s = SETS - 1; s >= s0; s--)
#pragma unroll
    for (int r = 0; r < kRows; r += 4) {
      if (s == set)
        fmac_self4<lk>(a[s][r], a[s][r + 1], a[s][r + 2], a[s][r + 3], -f[s]);
      else
        fmac_bcast4<lk>(a[s][r], a[s][r + 1], a[s][r + 2], a[s][r + 3], a[set][r], a[set][r + 1], a[set][r + 2],
                        a[set][r + 3], -f[s], -f[s], -f[s], -f[s]);
    }
  b[0] -= xb.x * fb;
  b[1] -= xb.y * fb;
}

template <int K, int NW, int SETS>
__device__ __forceinline__ void gels_steps(float (&a)[SETS][kRows], float (&b)[2], int t, int n, GelsLds<NW>& L) {
  if constexpr (K < 16 * SETS) {
    if (K >= n) return;  // uniform
    gels_step<K, NW, SETS>(a, b, t, L);
    gels_steps<K + 1, NW, SETS>(a, b, t, n, L);
  }
}

// NW wavefronts hold 128 NW rows at a time; a taller problem goes through in
// chunks, the triangle and Q^T b of the rows so far as the next chunk's first
// 32 rows (a sequential TSQR).  SETS: 16-column register sets (n <= 16 SETS).
template <int NW, int SETS>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4)))
gels_kernel(int count, int m, int n, const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ X) {
  __shared__ GelsLds<NW> L;
  const int t = threadIdx.x, lane = t & 63;
  const int grp = t >> 4;  // row group
  constexpr int kChunk = 128 * NW;
  for (int p = blockIdx.x; p < count; p += gridDim.x) {
    // rows past m read 0 by the descriptors' range check
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(A + (int64_t)p * m * n), (short)0, 4 * m * n, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B + (int64_t)p * m), (short)0, 4 * m, 0x00020000);
    float a[SETS][kRows], b[2];
    int done = 0;  // rows factored so far
    for (;;) {
      // row group 0 of a later chunk is the triangle (rows 0..31), the rest new rows
      const bool tri = done > 0 && grp == 0;
      int c = lane & 15;
      asm volatile("" : "+v"(c));  // as in the steps
      const int row0 = done > 0 ? done + (grp - 1) * kRows : grp * kRows;
      if (tri) {
#pragma unroll
        for (int s = 0; s < SETS; s++)
#pragma unroll
          for (int r = 0; r < kRows; r++) {
            const int col = 16 * s + c;
            a[s][r] = r <= col && col < n ? L.R[r][col] : 0.f;
          }
#pragma unroll
        for (int i = 0; i < 2; i++) b[i] = 2 * c + i < n ? L.y[2 * c + i] : 0.f;
      } else {
#pragma unroll
        for (int s = 0; s < SETS; s++) {
          // columns past n start out of range and stay there (a row group's
          // offsets span 31 n elements, under 4 KB)
          uint32_t off = 16 * s + c < n ? 4u * ((uint32_t)row0 * (uint32_t)n + (uint32_t)(16 * s + c)) : 0x80000000u;
#pragma unroll
          for (int r = 0; r < kRows; r++, off += 4u * (uint32_t)n) a[s][r] = buf_load<float>(ra, off);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) b[i] = buf_load<float>(rb, 4u * (uint32_t)(row0 + 2 * c + i));
      }
      gels_steps<0, NW, SETS>(a, b, t, n, L);
      done += done > 0 ? kChunk - kRows : kChunk;
      if (done >= m) break;
      if (NW > 1) __syncthreads();  // the last step's sums are read before the next chunk's first are written
      else __builtin_amdgcn_wave_barrier();
    }
    // R x = (Q^T b)[0:n] in wavefront 0, a row per lane; the reciprocals of
    // the diagonal once for all lanes, each quotient corrected by its residual
    // (a division inside the chain costs four times as much; it is taken where
    // an entry of the diagonal has no finite reciprocal)
    if (t < 64) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      int i = lane & 31;
      asm volatile("" : "+v"(i));  // its lane masks are not worth keeping across problems
      const bool live = i < n;
      float rr[16 * SETS];
#pragma unroll
      for (int q = 0; q < 16 * SETS; q++) rr[q] = live && q >= i && q < n ? L.R[i][q] : 0.f;
      float acc = live ? L.y[i] : 0.f;
      const float diag = live ? L.R[i][i] : 1.f;
      const float inv = 1.f / diag;
      const bool divide = __ballot(!(fabsf(diag) >= 1e-37f)) != 0;
#pragma unroll
      for (int q = 16 * SETS - 1; q >= 0; q--) {
        if (q < n) {  // uniform
          float v = acc * inv;
          const float v2 = fmaf(fmaf(-v, diag, acc), inv, v);
          v = v2 == v2 ? v2 : v;  // an infinity stays one
          if (divide) v = acc / diag;  // uniform
          const float xq = readlane_f(v, q);
          if (i == q) acc = xq;
          else if (i < q) acc -= rr[q] * xq;
        }
      }
      if (lane < n) X[(int64_t)p * n + lane] = acc;
    }
    // the next problem's first sums go to the buffer that this one's last
    // step, when n is odd, may still be reading
    if (NW > 1) __syncthreads();
  }
}

template <int NW>
int gels_launch(nmx_ctx* ctx, int count, int m, int n, const float* A, const float* B, float* X) {
  // 128 registers a thread: 16 wavefronts of it fit a CU
  const int grid = std::min(count, ctx->num_cus * (16 / NW));
  if (n <= 16) gels_kernel<NW, 1><<<grid, 64 * NW, 0, ctx->stream>>>(count, m, n, A, B, X);
  else gels_kernel<NW, 2><<<grid, 64 * NW, 0, ctx->stream>>>(count, m, n, A, B, X);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

}  // namespace

NMX_API int nmx_batched_gels_f32(nmx_ctx* ctx, int count, int m, int n, const float* A, const float* B, float* X) {
  if (!ctx) return -1;
  if (count < 0) return -2;
  if (m < 1) return -3;
  if (n < 1 || n > 32 || n > m) return -4;
  if (count == 0) return NMX_OK;
  if (!A) return -5;
  if (!B) return -6;
  if (!X) return -7;
  if ((int64_t)m * n * 4 >= 0x7FFFFFFF) return NMX_ERR_UNSUPPORTED;
  ProfScope ps(ctx, K_TSQR, 0.0, 4.0 * (double)count * ((double)m * n + m + n));
  // the fewest wavefronts that hold the problem (128 rows each): a smaller
  // workgroup has a shorter step and more problems share a CU
  if (m <= 128) return gels_launch<1>(ctx, count, m, n, A, B, X);
  if (m <= 256) return gels_launch<2>(ctx, count, m, n, A, B, X);
  if (m <= 512) return gels_launch<4>(ctx, count, m, n, A, B, X);
  if (m <= 1024) return gels_launch<8>(ctx, count, m, n, A, B, X);
  return gels_launch<16>(ctx, count, m, n, A, B, X);
}
