// Batched symmetric eigensolver for small matrices (n <= 64), FP32: the
// register-tier `eigh` that numax's `map` runs one matrix per GPU thread
// (numax/linalg/_array/eigen.mojo:316-392, rotation :34-75), one wavefront
// segment per matrix here.
//
// numax sweeps the pairs (p, q) in cyclic-by-row order, one rotation at a
// time.  Rotations on disjoint pairs commute, so here every step rotates
// NP/2 disjoint neighbour pairs at once -- (0,1),(2,3),... on even steps,
// (1,2),(3,4),... on odd ones -- and each rotation also exchanges its two
// indices.  With the exchange every index travels one way through the
// ordering, so NP steps meet every pair exactly once (the odd-even
// transposition network), and all register indices stay static.  The
// rotation itself is numax's (_jacobi_rotation): t = sign(d) 2 a_pq /
// guard(|d| + sqrt(d^2 + 4 a_pq^2)), c = 1 / sqrt(1 + t^2), s = t c, with
// d = a_qq - a_pp, and the same fixed number of sweeps (12 by default, no
// convergence test).  The diagonal is carried separately (a_pp - t a_pq,
// a_qq + t a_pq), which is where the eigenvalues are read.  A different
// rotation order changes rounding, not the converged result: eigenvalues are
// compared sorted against the FP64 oracle.
//
// Layout: lane L of a segment of NP lanes holds column L of A and of V in
// registers (NP = 32 packs two matrices per wavefront, NP = 64 one); rows
// are register indices.  A matrix of order n < NP is padded with zero rows
// and columns, which only ever rotate by exact exchanges (a_pq = 0).
//
// What bounds it: vector issue, about 640 instructions a step of a 64-wide
// wavefront (192 for the rows of A, 320 for the columns of A and V, 90 for
// the rotation, 32 to pick a_pq).  A pair's lanes are neighbours, so the
// other lane's entry is a DPP operand of the multiply (quad_perm on even
// steps, wave_shl / wave_shr on odd ones) and the rotations reach the rows as
// broadcast LDS reads.  As lane shuffles through LDS, two a register row plus
// two a rotation, they bound the kernel: 65,536 matrices of order 24 to 64
// took 77.8 ms; they take 25.5 ms now, with the
// same eigenvalues bit for bit.
#include <math.h>

#include "nmx_internal.h"

namespace {

constexpr float kFloorF = 1e-30f;  // numax/linalg/common.mojo:27-29

__device__ __forceinline__ float guard_f(float x) {
  const float m = fabsf(x);
  return (m >= kFloorF || m != m) ? x : copysignf(kFloorF, x);
}

// v of the lane `CTRL` names (a DPP control; folds into the consuming instruction)
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
constexpr int kSwapPairs = 0xB1;  // quad_perm 1,0,3,2: lane ^ 1
constexpr int kFromNext = 0x130;  // wave_shl:1: lane + 1
constexpr int kFromPrev = 0x138;  // wave_shr:1: lane - 1

// x of the pair's other lane (OFF = 0: lane ^ 1; OFF = 1: lane + 1 on a first
// lane, lane - 1 on a second; lanes without a pair get any value)
template <int OFF>
__device__ __forceinline__ float other(float x, bool isP) {
  if constexpr (OFF == 0) return dpp<kSwapPairs>(x);
  // both on every lane: a DPP move reads lanes a branch would have turned off
  const float next = dpp<kFromNext>(x), prev = dpp<kFromPrev>(x);
  return isP ? next : prev;
}

// a[L+1] on every first lane L of a pair (lanes L = OFF, OFF+2, ... of each
// segment): the two candidates of each quad by lane parity, then the quads
// merged by bank-masked moves.
template <int NP, int OFF, int G = 0>
__device__ __forceinline__ float pick_next(const float (&a)[NP], bool upper, float x) {
  if constexpr (4 * G < NP) {
    constexpr int r0 = 4 * G + 1 + OFF, r1 = 4 * G + 3 + OFF;  // a[L+1] of the quad's two first lanes
    const float lo = a[r0], hi = a[r1 < NP ? r1 : NP - 1];
    const float cand = upper ? hi : lo;
    constexpr int row = G / 4;  // 16-lane row; with 32-lane segments the other segment's too
    constexpr int rows = NP == 64 ? 1 << row : (1 << row) | (1 << (row + 2));
    x = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(x), __float_as_int(cand), 0xE4, rows, 1 << (G % 4), false));
    return pick_next<NP, OFF, G + 1>(a, upper, x);
  } else {
    return x;
  }
}

// x := alpha x + beta (the pair's other lane's x) for four registers, the
// second product rounded first.  OFF = 1 adds both neighbours' products, one
// of which has a zero coefficient.  Written out because the compiler folds
// no DPP move into the second multiply-add; s_nop 1 gives the two wait states
// between a vector write and a DPP read of the same register.
template <int OFF>
__device__ __forceinline__ void rotate_col4(float& x0, float& x1, float& x2, float& x3, float alpha, float beta,
                                            float beta_next, float beta_prev) {
  float t0, t1, t2, t3;
  if constexpr (OFF == 0) {
    asm volatile(
        "s_nop 1\n"
        "v_mul_f32_dpp %4, %0, %9 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %5, %1, %9 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %6, %2, %9 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %7, %3, %9 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "v_fma_f32 %0, %8, %0, %4\n"
        "v_fma_f32 %1, %8, %1, %5\n"
        "v_fma_f32 %2, %8, %2, %6\n"
        "v_fma_f32 %3, %8, %3, %7\n"
        : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(alpha), "v"(beta));
  } else {
    asm volatile(
        "s_nop 1\n"
        "v_mul_f32_dpp %4, %0, %10 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_mul_f32_dpp %5, %1, %10 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_mul_f32_dpp %6, %2, %10 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_mul_f32_dpp %7, %3, %10 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_fmac_f32_dpp %4, %0, %9 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_fmac_f32_dpp %5, %1, %9 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_fmac_f32_dpp %6, %2, %9 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_fmac_f32_dpp %7, %3, %9 wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n"
        "v_fma_f32 %0, %8, %0, %4\n"
        "v_fma_f32 %1, %8, %1, %5\n"
        "v_fma_f32 %2, %8, %2, %6\n"
        "v_fma_f32 %3, %8, %3, %7\n"
        : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(alpha), "v"(beta_next), "v"(beta_prev));
  }
}

// A rotated and exchanged pair of rows (r, r + 1): p = s x + c y, q = c x - s y.
// Which product is rounded first is written out, here and above: equal
// diagonals rotate by the sign of a rounding error, so the order in which the
// eigenvalues come out follows it.  The six pairs that round c y first keep
// the order these results have had since the kernel's first build: with one
// rule for all pairs some 500 of the 2.75 million eigenvalues of 65,536
// matrices, half of them symmetric wells, come out in another place.
template <int NP, int OFF>
__device__ __forceinline__ void rotate_row(int r, float& p, float& q, float x, float y, float c, float s) {
  const bool cy_first = NP == 64 && OFF == 1 && r >= 13 && r <= 23;
  p = cy_first ? __builtin_fmaf(s, x, c * y) : __builtin_fmaf(c, y, s * x);
  q = __builtin_fmaf(c, x, -(s * y));
}

// The columns of V, eight rows at a time while they hold rows below nmax
// (uniform).  Recursive, so that every register index is a constant early.
template <int NP, int OFF, int I0>
__device__ __forceinline__ void rotate_rows(float (&v)[NP], int nmax, float alpha, float beta, float beta_next,
                                            float beta_prev) {
  if constexpr (I0 < NP) {
    if (I0 < nmax) {
#pragma unroll
      for (int i = I0; i < I0 + 8; i += 4)
        rotate_col4<OFF>(v[i], v[i + 1], v[i + 2], v[i + 3], alpha, beta, beta_next, beta_prev);
    }
    rotate_rows<NP, OFF, I0 + 8>(v, nmax, alpha, beta, beta_next, beta_prev);
  }
}

// One step of the ordering: rotate the pairs (OFF, OFF+1), (OFF+2, OFF+3),
// ... of every segment, exchanging the two indices of each pair.  cs: this
// segment's NP/2 rotations in LDS.
template <int NP, int OFF>
__device__ __forceinline__ void jacobi_step(float (&a)[NP], float (&v)[NP], float& d, int& player, int L, int nmax,
                                            float2* cs) {
  const bool odd = L & 1;
  const bool isP = OFF == 0 ? !odd : (odd && L + 1 < NP);
  const bool isQ = OFF == 0 ? odd : (!odd && L >= 1);
  // the pair's rotation, computed on its first lane (_array/eigen.mojo:34-75)
  const float apq_own = pick_next<NP, OFF>(a, L & 2, 0.f);  // a[L+1][L]: a_pq on a first lane
  const float d_next = OFF == 0 ? dpp<kSwapPairs>(d) : dpp<kFromNext>(d);
  float c, s, t;
  {
    const float twice = 2.f * apq_own;
    const float den = d_next - d;
    const float radius = sqrtf(__builtin_fmaf(twice, twice, den * den));
    const float safe = guard_f(fabsf(den) + radius);
    t = copysignf(1.f, den) * twice / safe;
    c = 1.f / sqrtf(__builtin_fmaf(t, t, 1.f));
    s = t * c;
  }
  if (isP) cs[L >> 1] = make_float2(c, s);
  wave_lds_order();
  const float c_o = other<OFF>(c, isP), s_o = other<OFF>(s, isP), t_o = other<OFF>(t, isP);
  const float apq_o = other<OFF>(apq_own, isP), d_o = other<OFF>(d, isP);
  if (isQ) {
    c = c_o;
    s = s_o;
    t = t_o;
  }
  const float apq = isQ ? apq_o : apq_own;
  // diagonal after the rotation and the exchange
  const float d_new = isP || isQ ? __builtin_fmaf(isP ? t : -t, apq, isP ? d_next : d_o) : d;
  // rows: register pairs (r, r+1), r = OFF, OFF+2, ... (every column); the
  // rotations come two pairs to a broadcast LDS read
#pragma unroll
  for (int r = OFF; r + 1 < NP; r += 4) {
    const float4 w = *(const float4*)(cs + (r >> 1));  // c, s of pairs r and r + 2
    {
      const float x = a[r], y = a[r + 1];
      rotate_row<NP, OFF>(r, a[r], a[r + 1], x, y, w.x, w.y);
    }
    if (r + 3 < NP) {
      const float x = a[r + 2 < NP ? r + 2 : 0], y = a[r + 3 < NP ? r + 3 : 0];
      rotate_row<NP, OFF>(r + 2, a[r + 2 < NP ? r + 2 : 0], a[r + 3 < NP ? r + 3 : 0], x, y, w.z, w.w);
    }
  }
  wave_lds_order();
  // columns of A and V (with the exchange): new = alpha own + beta partner's.
  // Lanes without a pair sit out: beside one may be another matrix's lane, and
  // a zero coefficient does not keep its infinities and NaNs out.  (What a
  // neighbour reads of a lane that sits out is 0.)
  const float alpha = isP ? s : -s;
  const float beta_next = isP ? c : 0.f, beta_prev = isQ ? c : 0.f;
  if (OFF == 0 || isP || isQ) {
#pragma unroll
    for (int i = 0; i < NP; i += 4)
      rotate_col4<OFF>(a[i], a[i + 1], a[i + 2], a[i + 3], alpha, c, beta_next, beta_prev);
    // V's rows past the matrix's order are never read
    rotate_rows<NP, OFF, 0>(v, nmax, alpha, c, beta_next, beta_prev);
  }
  d = d_new;
  const int player_o = __float_as_int(other<OFF>(__int_as_float(player), isP));
  player = isP || isQ ? player_o : player;
}

struct EighArgs {
  int count;
  const int32_t* n;
  const int64_t* offA;  // matrix (and vectors) element offset
  const int64_t* offW;  // eigenvalue offset
  const float* A;
  float* W;
  float* V;             // nullable
  int sweeps;
  const int32_t* order;
  const int32_t* cls;   // [0] begin / [1] count for NP = 32, [2] / [3] for NP = 64
  int32_t* head;
};

template <int NP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NP == 64 ? 2 : 4)))
syevj_kernel(EighArgs args, int cls) {
  constexpr int PPW = 64 / NP;  // matrices per wavefront
  __shared__ __attribute__((aligned(16))) float2 rot[256 / NP][NP / 2];
  const int lane = threadIdx.x & 63;
  const int L = lane & (NP - 1);       // slot within the segment
  float2* cs = rot[threadIdx.x / NP];
  const int seg = lane / NP;
  const int begin = args.cls[2 * cls], count = args.cls[2 * cls + 1];

  for (;;) {
    int slot0 = 0;
    if (lane == 0) slot0 = atomicAdd(&args.head[cls], PPW);
    slot0 = __shfl(slot0, 0);
    if (slot0 >= count) break;
    const int slot = slot0 + seg;
    const bool live = slot < count;
    const int p = live ? args.order[begin + slot] : 0;
    const int n = live ? args.n[p] : 0;
    const float* A = args.A + (live ? args.offA[p] : 0);
    // V rows a wavefront needs: the larger of its matrices' orders
    const int nmax = NP == 64 ? n : max(n, __shfl_xor(n, 32));
    float a[NP], v[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
      a[i] = (i < n && L < n) ? A[(int64_t)i * n + L] : 0.f;
      v[i] = (i == L) ? 1.f : 0.f;
    }
    float d = L < n ? A[(int64_t)L * n + L] : 0.f;
    int player = L;

    for (int sw = 0; sw < args.sweeps; sw++) {
#pragma unroll 1
      for (int step = 0; step < NP; step += 2) {
        jacobi_step<NP, 0>(a, v, d, player, L, __builtin_amdgcn_readfirstlane(nmax), cs);
        jacobi_step<NP, 1>(a, v, d, player, L, __builtin_amdgcn_readfirstlane(nmax), cs);
      }
    }
    // padding players (>= n) only ever exchanged; each real player's value
    // and vector go to its own index
    if (live && player < n) {
      args.W[args.offW[p] + player] = d;
      if (args.V) {
        float* V = args.V + args.offA[p];
#pragma unroll
        for (int i = 0; i < NP; i++)
          if (i < n) V[(int64_t)i * n + player] = v[i];
      }
    }
  }
}

// A matrix is taken when 1 <= n <= 64 and its matrix and eigenvalues lie
// inside the arrays the caller sized; others are skipped.
__device__ __forceinline__ bool eigh_ok(int nn, int64_t oa, int64_t ow, int64_t a_elems, int64_t w_elems) {
  return nn >= 1 && nn <= 64 && oa >= 0 && oa + (int64_t)nn * nn <= a_elems && ow >= 0 && ow + nn <= w_elems;
}

__global__ void eigh_sort_kernel(int count, const int32_t* __restrict__ n, const int64_t* __restrict__ offA,
                                 const int64_t* __restrict__ offW, int64_t a_elems, int64_t w_elems,
                                 int32_t* __restrict__ cls, int32_t* __restrict__ order, int32_t* __restrict__ head) {
  // one workgroup: counts, then a stable scatter by class (n <= 32 first)
  __shared__ int cnt[2];
  const int t = threadIdx.x;
  if (t < 2) cnt[t] = 0;
  __syncthreads();
  for (int i = t; i < count; i += blockDim.x) {
    const int nn = n[i];
    if (eigh_ok(nn, offA[i], offW[i], a_elems, w_elems)) atomicAdd(&cnt[nn > 32], 1);
  }
  __syncthreads();
  if (t == 0) {
    cls[0] = 0;
    cls[1] = cnt[0];
    cls[2] = cnt[0];
    cls[3] = cnt[1];
    head[0] = 0;
    head[1] = 0;
    cnt[0] = 0;
    cnt[1] = 0;
  }
  __syncthreads();
  for (int i = t; i < count; i += blockDim.x) {
    const int nn = n[i];
    if (eigh_ok(nn, offA[i], offW[i], a_elems, w_elems)) {
      const int c = nn > 32;
      order[cls[2 * c] + atomicAdd(&cnt[c], 1)] = i;
    }
  }
}

}  // namespace

NMX_API int nmx_batched_syevj_f32(nmx_ctx* ctx, int count, const int32_t* n, const int64_t* offA,
                                  const int64_t* offW, const float* A, int64_t a_elems, float* W, int64_t w_elems,
                                  float* V, int sweeps) {
  if (!ctx) return -1;
  if (count < 0) return -2;
  if (count == 0) return NMX_OK;
  if (!n) return -3;
  if (!offA) return -4;
  if (!offW) return -5;
  if (!A) return -6;
  if (a_elems <= 0) return -7;
  if (!W) return -8;
  if (w_elems <= 0) return -9;
  if (sweeps < 0) return -11;
  void* ws = nullptr;
  NMX_TRY(nmx_workspace(ctx, sizeof(int32_t) * (8 + (size_t)count), &ws));
  int32_t* cls = (int32_t*)ws;
  int32_t* head = cls + 4;
  int32_t* order = cls + 8;
  {
    ProfScope ps(ctx, K_OTHER, 0.0, 0.0);
    eigh_sort_kernel<<<1, 1024, 0, ctx->stream>>>(count, n, offA, offW, a_elems, w_elems, cls, order, head);
    NMX_HIP(ctx, hipGetLastError());
  }
  EighArgs a{count, n, offA, offW, A, W, V, sweeps, order, cls, head};
  {
    ProfScope ps(ctx, K_EIGH, 0.0, 0.0);
    const int grid = ctx->num_cus * 4;
    syevj_kernel<64><<<grid, 256, 0, ctx->stream>>>(a, 1);
    syevj_kernel<32><<<grid, 256, 0, ctx->stream>>>(a, 0);
    NMX_HIP(ctx, hipGetLastError());
  }
  return NMX_OK;
}
