// Panel kernels of the blocked factorizations: the cooperative pivoting leaf,
// row interchanges, the recursion of the triangular solves, and the small
// gather / tril helpers.
//
// numax runs its panels as single-workgroup kernels over the whole remaining
// height (numax/linalg/panel.mojo:289-431) while the rest of the device idles;
// its own docstring names that as the ceiling (panel.mojo:41-49).  Here the
// leaf of the recursive panel is spread over up to 32 workgroups of 512
// threads, one matrix row per thread held in registers (two above 16384 rows),
// and the per-column pivot search is one exchange through a mailbox in device
// memory; up to 1024 rows one workgroup holds them all.
#include <limits.h>

#include "tile16.h"

namespace {

constexpr double kPivotFloor = 1e-30;  // numax/linalg/common.mojo:27-29
constexpr long kSpinLimit = 1L << 23;  // bounded waits: a few seconds at worst

// ---- mailbox ----------------------------------------------------------------
// Every word a participant publishes is a 64-bit atomic holding 32 bits of
// payload and the 32-bit epoch of the column it belongs to, so a reader
// validates each word on its own and needs no fence and no second trip.  A
// double travels as two words.  Slots are double-buffered by epoch parity: a
// participant can only publish column j+2 after every participant has
// published j+1, which each does only after reading all of column j.
template <typename T>
struct MbLayout {
  static constexpr int VW = sizeof(T) / 4;       // words per value
  static constexpr int STRIDE = 1 + VW + kLeafW * VW;  // header, |pivot|, row values
  static constexpr int PARITY = kMaxParts * STRIDE;
};
static_assert(2 * MbLayout<double>::PARITY * 8 <= kMailboxBytes, "mailbox too small");

__device__ __forceinline__ uint64_t mb_pack(uint32_t payload, uint32_t epoch) {
  return ((uint64_t)payload << 32) | epoch;
}
__device__ __forceinline__ void mb_put(uint64_t* w, uint32_t payload, uint32_t epoch) {
  __hip_atomic_store(w, mb_pack(payload, epoch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Pivot keys: a candidate's magnitude as its (order-preserving) bit pattern
// plus one, 0 for "no candidate".  Equal keys are equal magnitudes, so the
// first maximum is the smallest row among the largest key.
template <typename T>
struct PivKey;
template <>
struct PivKey<float> {
  typedef uint32_t K;
  static __device__ __forceinline__ K of(float mag) { return __float_as_uint(mag) + 1u; }
  static constexpr int WORDS = 1;
  static __device__ __forceinline__ uint32_t word(K k, int i) { return k; }
  static __device__ __forceinline__ K from(const uint32_t* w) { return w[0]; }
};
template <>
struct PivKey<double> {
  typedef uint64_t K;
  static __device__ __forceinline__ K of(double mag) { return (uint64_t)__double_as_longlong(mag) + 1ull; }
  static constexpr int WORDS = 2;
  static __device__ __forceinline__ uint32_t word(K k, int i) { return i ? (uint32_t)(k >> 32) : (uint32_t)k; }
  static __device__ __forceinline__ K from(const uint32_t* w) { return ((uint64_t)w[1] << 32) | w[0]; }
};

// ---------------------------------------------------------------------------
// Cooperative leaf of the recursive LU panel.
//
// Factors columns c0..c0+w (w <= 32) over rows r0..n with partial pivoting,
// exactly getrf_panel's arithmetic (panel.mojo:289-431): first-maximum pivot
// (ties to the lower row; the diagonal row counts as magnitude >= 0, so an
// all-zero or all-NaN column keeps its diagonal; NaN never wins),
// interchange, an exact-zero pivot divided as 1e-30 with `info` recording the
// first, correctly rounded quotients for the multipliers and the rank-1
// update of the panel's own columns, every multiply-add fused.  The leaf's
// interchanges are then replayed over every other column of the matrix right
// after (laswp_gather_kernel), which leaves the matrix numax's full-width
// swaps leave (panel.mojo:404-411).
//
// Workgroup p of `parts` owns rows r0 + 512 ROWS p + t + 512 i (i < ROWS) of
// its threads (alone, up to 1024 rows of as many threads), each row's 32
// columns in registers.  Rows stay where they are:
// a thread keeps the position its row has in the interchanged panel and
// stores it there at the end.  The columns are walked in groups of eight with
// the registers rotated by eight after each, so that within a group every
// register index is static and the loop over groups (and the instruction
// cache) stays short.  Per column, in one workgroup: a DPP maximum of the
// pivot key's high word (its low word and the position only where that ties),
// each wavefront's winning row staged in LDS, one barrier.  Across workgroups
// (parts > 1, grid 8 * parts of which every eighth takes part, so all
// participants share one XCD and its L2): each part publishes its winner and
// key as epoch-tagged 64-bit words, and every thread of every part spins on
// the words it stages, no fences: all of them in one round trip up to 16
// parts; above that the keys and positions first, then the winner's row.
// Slots alternate by epoch parity: a part publishes column j+2 only after
// reading every part's key for column j+1, which each part publishes only
// after its reads of column j.
//
// What bounds it: the chain of one pivot decision per column.  Rotated by one
// register a column, with every column's update and select run to full width,
// both rows physically swapped through LDS and three maxima a decision, a
// column took 3.7 us (1000 rows FP64, one workgroup) and 4.0 us (8192 rows,
// sixteen); it takes 1.6 us (mean over 1000 .. 32 rows) and 2.9 us.
// An FP64 quotient is the product with the pivot's reciprocal and two
// corrections: one correction leaves rare last bits wrong, which a system of
// condition 1e6 carries into x, and saves 1.4 of a 32-column leaf's 91.6 us
// (order 8192, mean over its panels).
// ---------------------------------------------------------------------------
constexpr int kLeafT = 512;      // threads per workgroup of several
constexpr int kLeafMaxT = 1024;  // threads at most, in a workgroup alone
constexpr int kTwoPhaseParts = 16;  // above this many parts the exchange reads the winner's row only
constexpr int kLeafWaves = kLeafMaxT / 64;
constexpr int kLeafG = 8;    // columns a group

// The lane with the largest key, the smallest position among equals; key 0
// everywhere gives some lane.  All arguments per lane, the result uniform.
__device__ __forceinline__ int winner_lane(uint64_t key, int pos) {
  const uint32_t khi = (uint32_t)(key >> 32);
  const uint32_t hi = wave_umax(khi);
  uint64_t m = __ballot(khi == hi);
  if (m & (m - 1)) {  // uniform
    const uint32_t lo = wave_umax(khi == hi ? (uint32_t)key : 0u);
    const bool eq = khi == hi && (uint32_t)key == lo;
    m = __ballot(eq);
    if (m & (m - 1)) {
      const uint32_t p = wave_umin(eq ? (uint32_t)pos : 0xFFFFFFFFu);
      m = __ballot(eq && (uint32_t)pos == p);
    }
  }
  return __ffsll((long long)m) - 1;
}
__device__ __forceinline__ int winner_lane(uint32_t key, int pos) {
  const uint32_t k = wave_umax(key);
  uint64_t m = __ballot(key == k);
  if (m & (m - 1)) {  // uniform
    const uint32_t p = wave_umin(key == k ? (uint32_t)pos : 0xFFFFFFFFu);
    m = __ballot(key == k && (uint32_t)pos == p);
  }
  return __ffsll((long long)m) - 1;
}
__device__ __forceinline__ uint32_t key_at(uint32_t k, int lane) { return __builtin_amdgcn_readlane(k, lane); }
__device__ __forceinline__ uint64_t key_at(uint64_t k, int lane) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((uint32_t)(k >> 32), lane) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((uint32_t)k, lane);
}

// The same over lanes 0..15 only (one candidate a wavefront).
__device__ __forceinline__ uint32_t row_umax(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false));
  return __builtin_amdgcn_readlane(v, 0);
}
__device__ __forceinline__ uint32_t key_high(uint32_t k) { return k; }
__device__ __forceinline__ uint32_t key_high(uint64_t k) { return (uint32_t)(k >> 32); }
template <typename K>
__device__ __forceinline__ int winner_lane16(K key, int pos) {
  const uint32_t hi = row_umax(key_high(key));
  const uint64_t m = __ballot(key_high(key) == hi) & 0xFFFFull;
  if (m & (m - 1)) return winner_lane(key, pos);  // uniform; the lanes above hold no key
  return __ffsll((long long)m) - 1;
}

template <typename T>
struct LeafLds {
  static constexpr int W = kLeafW, VW = MbLayout<T>::VW;
  typedef typename PivKey<T>::K Key;
  // staged mailbox words, per part [values | key | position] (PSTRIDE even, so
  // every part's values stay 8-byte aligned)
  static constexpr int PSTRIDE = (W * VW + VW + 1 + 1) & ~1;
  // double-buffered by column parity
  __attribute__((aligned(16))) T slot_v[2][kLeafWaves][W];  // each wavefront's winning row
  Key slot_k[2][kLeafWaves];
  int slot_p[2][kLeafWaves];
  __attribute__((aligned(16))) uint32_t stage[2][kMaxParts * PSTRIDE];
  int aborted, info_set;
};

struct LeafArgs {
  int n, r0, c0, w, parts, p;  // p: this workgroup's part
  int32_t* ipiv;
  int32_t* info;
  uint64_t* mb;
  uint32_t epoch0;
};

// Column S of the group that starts at leaf column jb.
template <int S, typename T, int ROWS, bool MULTI>
__device__ __forceinline__ void leaf_step(const LeafArgs& a, T (&v)[ROWS][kLeafW], int (&pos)[ROWS], int jb, int nwaves,
                                          LeafLds<T>& L) {
  constexpr int W = kLeafW, VW = MbLayout<T>::VW, STRIDE = MbLayout<T>::STRIDE, PSTRIDE = LeafLds<T>::PSTRIDE;
  typedef PivKey<T> PK;
  typedef typename PK::K Key;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int j = jb + S, gr = a.r0 + j, gc = a.c0 + j, par = j & 1;

  // 1. this thread's candidate: largest key, smallest position
  Key tk = 0;
  int tp = INT_MAX, ti = 0;
#pragma unroll
  for (int i = 0; i < ROWS; i++) {
    T mag = fabs(v[i][S]);
    if (!(mag == mag)) mag = T(-1);               // NaN never wins ...
    if (pos[i] == gr && mag < T(0)) mag = T(0);   // ... the diagonal row starts at 0
    const bool cand = pos[i] >= gr && pos[i] < a.n && mag >= T(0);
    const Key k = cand ? PK::of(mag) : Key(0);
    if (k > tk || (k == tk && k != 0 && pos[i] < tp)) {
      tk = k;
      tp = pos[i];
      ti = i;
    }
  }
  // 2. the wavefront's, and its row into LDS
  const int wl = winner_lane(tk, tp);
  if (lane == wl) {
#pragma unroll
    for (int i = 0; i < ROWS; i++)
      if (ROWS == 1 || i == ti) {
        // from this column on (finished columns stay with their rows)
#pragma unroll
        for (int g = 0; g < W / kLeafG; g++)
          if (g == 0 || jb + kLeafG * g < a.w) {  // uniform
#pragma unroll
            for (int c = g ? 0 : S; c < kLeafG; c++) L.slot_v[par][wave][kLeafG * g + c] = v[i][kLeafG * g + c];
          }
      }
    L.slot_k[par][wave] = tk;
    L.slot_p[par][wave] = tp;
  }
  __syncthreads();
  // 3. the workgroup's winner (every wavefront works it out)
  Key ck = 0;
  int cp = INT_MAX;
  if (lane < nwaves) {
    ck = L.slot_k[par][lane];
    cp = L.slot_p[par][lane];
  }
  const int gw = winner_lane16(ck, cp);
  int wp = __builtin_amdgcn_readlane(cp, gw);
  const T* urow = L.slot_v[par][gw];
  if constexpr (MULTI) {
    const uint32_t epoch = a.epoch0 + (uint32_t)j + 1u;
    const Key gk = key_at(ck, gw);
    // 4. publish this part's winner (or "none")
    uint64_t* mbp = a.mb + (size_t)(epoch & 1u) * MbLayout<T>::PARITY;
    uint64_t* myslot = mbp + (size_t)a.p * STRIDE;
    if (t < W * VW) {
      const uint32_t* src = (const uint32_t*)urow;
      mb_put(myslot + 1 + VW + t, gk != 0 ? src[t] : 0u, epoch);
    } else if (t < W * VW + VW) {
      mb_put(myslot + 1 + (t - W * VW), PK::word(gk, t - W * VW), epoch);
    } else if (t == W * VW + VW) {
      mb_put(myslot, (uint32_t)wp, epoch);
    }
    // 5. stage the parts' words, each validated by its epoch.  With many
    // parts every workgroup reading every part's whole row crowds the few
    // L2 lines they sit in, so it reads the keys and positions first, then
    // only the winner's values (two round trips, a tenth of the data; 10%
    // faster over a 32-part leaf, 2% slower over 8 parts).
    uint32_t* stg = L.stage[par];
    const bool two_phase = a.parts > kTwoPhaseParts;  // uniform
    auto stage_word = [&](const uint64_t* src, int dst) {
      uint64_t wv;
      long spins = 0;
      for (;;) {
        wv = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)wv == epoch) break;
        if (L.aborted || ++spins > kSpinLimit) { L.aborted = 1; break; }
        __builtin_amdgcn_s_sleep(1);
      }
      stg[dst] = (uint32_t)(wv >> 32);
    };
    // a slot's words still of use: its header and the columns ahead, which are
    // the first registers.  (A thread's words polled together instead of one
    // after the other crowd the same lines: 3.4 us a column against 3.0.)
    const int words = 1 + VW + min(W, (a.w - jb + kLeafG - 1) / kLeafG * kLeafG) * VW;
    if (two_phase) {
      constexpr int HW = VW + 1;  // header words of a slot: position, key
      for (int idx = t; idx < a.parts * HW; idx += kLeafT) {
        const int q = idx / HW, f = idx % HW;
        stage_word(mbp + (size_t)q * STRIDE + f, q * PSTRIDE + (f == 0 ? W * VW + VW : W * VW + f - 1));
      }
    } else {
      for (int idx = t; idx < a.parts * STRIDE; idx += kLeafT) {
        const int q = idx / STRIDE, f = idx % STRIDE;  // mailbox slot: [position | key | values]
        if (f < words)
          stage_word(mbp + idx, q * PSTRIDE + (f == 0 ? W * VW + VW : (f <= VW ? W * VW + f - 1 : f - 1 - VW)));
      }
    }
    __syncthreads();
    // 6. the global winner (lane q reads part q's; parts <= 32)
    Key pk = 0;
    int pp = INT_MAX;
    if (lane < a.parts) {
      const uint32_t* sq = stg + lane * PSTRIDE;
      pk = PK::from(sq + W * VW);
      pp = (int)sq[W * VW + VW];
    }
    const int bp = winner_lane(pk, pp);
    wp = __builtin_amdgcn_readlane(pp, bp);
    if (two_phase) {
      for (int idx = t; idx < W * VW; idx += kLeafT)
        stage_word(mbp + (size_t)bp * STRIDE + 1 + VW + idx, bp * PSTRIDE + idx);
      __syncthreads();
    }
    urow = (const T*)(stg + bp * PSTRIDE);
    // an exchange that gave up: any in-range row, the context reports it
    if (L.aborted) wp = gr;
  }
  // 7. the winner's row takes position gr, the row that had it the winner's
#pragma unroll
  for (int i = 0; i < ROWS; i++) pos[i] = pos[i] == wp ? gr : (pos[i] == gr ? wp : pos[i]);
  T pivot = urow[S];
  if (t == 0 && a.p == 0) {
    a.ipiv[gc] = wp;
    if (fabs(pivot) == T(0) && !L.info_set) {
      *a.info = gc + 1;
      L.info_set = 1;
    }
  }
  if (pivot == T(0)) pivot = T(kPivotFloor);
  // 8. multipliers and the rank-1 update of the leaf's remaining columns:
  // the rest of this group, then the groups that are still ahead (the others
  // hold finished columns)
  bool live[ROWS];
  T l[ROWS];
  // FP32 divides; FP64 too where an operand is out of the plain range
  bool divide = sizeof(T) == 4 || !plain_divisor(pivot);  // uniform
  if constexpr (sizeof(T) == 8) {
    const T rinv = reciprocal(pivot);
    bool odd = false;
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
      live[i] = pos[i] > gr && pos[i] < a.n;
      const T x = v[i][S];
      odd = odd || (live[i] && !plain_dividend(x));
      const T q = plain_quotient(x, pivot, rinv);
      l[i] = x == T(0) ? x * rinv : q;  // a zero keeps its sign
    }
    divide = divide || __ballot(odd) != 0;
  }
  if (divide) {
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
      live[i] = pos[i] > gr && pos[i] < a.n;
      l[i] = v[i][S] / pivot;
    }
  }
#pragma unroll
  for (int i = 0; i < ROWS; i++) v[i][S] = live[i] ? l[i] : v[i][S];
#pragma unroll
  for (int g = 0; g < W / kLeafG; g++) {
    if (g == 0 || jb + kLeafG * g < a.w) {  // uniform
      T u[kLeafG];
#pragma unroll
      for (int c = 0; c < kLeafG; c++)
        if (g > 0 || c > S) u[c] = urow[kLeafG * g + c];
#pragma unroll
      for (int i = 0; i < ROWS; i++) {
        if (live[i]) {
#pragma unroll
          for (int c = 0; c < kLeafG; c++)
            if (g > 0 || c > S) v[i][kLeafG * g + c] = v[i][kLeafG * g + c] - l[i] * u[c];
        }
      }
    }
  }
}

template <int S, typename T, int ROWS, bool MULTI>
__device__ __forceinline__ void leaf_group(const LeafArgs& a, T (&v)[ROWS][kLeafW], int (&pos)[ROWS], int jb, int nwaves,
                                           LeafLds<T>& L) {
  if constexpr (S < kLeafG) {
    if (jb + S < a.w) {  // uniform
      leaf_step<S, T, ROWS, MULTI>(a, v, pos, jb, nwaves, L);
      leaf_group<S + 1, T, ROWS, MULTI>(a, v, pos, jb, nwaves, L);
    }
  }
}

// One row per thread (ROWS 1) for a panel of up to 1024 rows in one
// workgroup or up to 32 x 512 rows over several (MULTI); two above that.
template <typename T, int ROWS, bool MULTI>
__global__ void __launch_bounds__(MULTI ? kLeafT : kLeafMaxT) getf2_leaf(T* __restrict__ A, int lda, int n, int r0, int c0, int w,
                                                     int32_t* __restrict__ ipiv, int32_t* __restrict__ info,
                                                     uint64_t* __restrict__ mb, uint32_t epoch0, int parts, int* err) {
  constexpr int W = kLeafW;
  if (MULTI && (blockIdx.x % kXcds) != 0) return;
  const int p = MULTI ? (int)(blockIdx.x / kXcds) : 0;
  const int t = threadIdx.x;
  __shared__ LeafLds<T> L;
  if (t == 0) {
    L.aborted = 0;
    L.info_set = (*info != 0);
  }
  const int first = r0 + p * (kLeafT * ROWS);  // row i of the thread: first + t + 512 i
  T v[ROWS][W];
  int pos[ROWS];
  {
    // one descriptor at this workgroup's first row: offsets stay below 1024 rows
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(A + (int64_t)first * lda + c0);
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
      pos[i] = first + t + kLeafT * i;
      const bool own = pos[i] < n;
      const uint32_t rel = (uint32_t)(t + kLeafT * i) * (uint32_t)lda;
#pragma unroll
      for (int c = 0; c < W; c++)
        v[i][c] = buf_load<T>(rs, (own & (c < w)) ? (rel + c) * (uint32_t)sizeof(T) : kBufOob);
    }
  }
  // every load has landed before this part publishes anything (see the stores)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  const LeafArgs a{n, r0, c0, w, parts, p, ipiv, info, mb, epoch0};
  const int nwaves = blockDim.x / 64;
#pragma unroll 1
  for (int jb = 0; jb < W; jb += kLeafG) {
    leaf_group<0, T, ROWS, MULTI>(a, v, pos, jb, nwaves, L);
    // the next group's columns to the front (four turns bring the first back)
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
      T head[kLeafG];
#pragma unroll
      for (int c = 0; c < kLeafG; c++) head[c] = v[i][c];
#pragma unroll
      for (int c = 0; c + kLeafG < W; c++) v[i][c] = v[i][c + kLeafG];
#pragma unroll
      for (int c = 0; c < kLeafG; c++) v[i][W - kLeafG + c] = head[c];
    }
  }
  if (L.aborted && t == 0) atomicExch(err, NMX_ERR_SYNC_TIMEOUT);
  // Rows change places across workgroups: no row is stored before every part
  // has loaded its own.  A part that has staged every part's words of the
  // first column knows that (each published them after its loads).
#pragma unroll
  for (int i = 0; i < ROWS; i++) {
    if (first + t + kLeafT * i < n) {
      T* dst = A + (int64_t)pos[i] * lda + c0;
#pragma unroll
      for (int c = 0; c < W; c++)
        if (c < w) dst[c] = v[i][c];
    }
  }
}

// Replay the interchanges ipiv[k1..k2) (k2 - k1 <= 32) over the columns
// [col_lo, col_hi) minus [skip_lo, skip_lo + skip_w): laswp / laswp_matrix
// (numax/linalg/panel.mojo:1824-1852, :2279-2313).  The net effect of the
// sequence on the <= 2(k2-k1) rows it touches is worked out once per
// workgroup in LDS; each thread then moves one column with all its loads in
// flight together.
template <typename T>
__global__ void __launch_bounds__(256) laswp_gather_kernel(T* __restrict__ A, int lda, int col_lo, int ncols,
                                                           int skip_lo, int skip_w, const int32_t* __restrict__ ipiv,
                                                           int k1, int k2) {
  __shared__ int mv_dst[2 * kLeafW], mv_src[2 * kLeafW], mv_count;
  const int t = threadIdx.x;
  const int w = k2 - k1;
  if (t < 64) {
    // wavefront 0: lane e tracks involved row e and the original row now in it
    int myrow = (t < w) ? k1 + t : -1;
    int mine = myrow;
    int nr = w;
    // the pivots once, one per lane (a load inside the walk waited a scalar
    // round trip per step)
    const int qv = t < w ? ipiv[k1 + t] : 0;
    for (int j = 0; j < w; j++) {
      const int q = __builtin_amdgcn_readlane(qv, j);
      const unsigned long long hit = __ballot(t < nr && myrow == q);
      int pos;
      if (hit) {
        pos = __ffsll((long long)hit) - 1;
      } else {
        pos = nr;
        if (t == nr) { myrow = q; mine = q; }
        nr++;
      }
      // j and pos are the same in every lane: v_readlane, where a shuffle
      // would go through LDS twice a step (10.3 -> 9.5 us a launch at order 1000)
      const int cj = __builtin_amdgcn_readlane(mine, j);
      const int cp = __builtin_amdgcn_readlane(mine, pos);
      if (t == j) mine = cp;
      if (t == pos) mine = cj;
    }
    const bool moved = (t < nr) && (mine != myrow);
    const unsigned long long mm = __ballot(moved);
    if (moved) {
      const int at = __popcll(mm & ((1ull << t) - 1ull));
      mv_dst[at] = myrow;
      mv_src[at] = mine;
    }
    if (t == 0) mv_count = __popcll(mm);
  }
  __syncthreads();
  const int moves = mv_count;
  if (moves == 0) return;
  // lane e of each wavefront takes move e out of LDS (one read), and every
  // move's rows then come to the whole wavefront by v_readlane: read per
  // move, the list cost one LDS round trip ahead of each load.  Every lane
  // stays active to the end (v_readlane reads lanes the branch would have
  // turned off); lanes past the last column load from the first one and
  // store nothing.
  static_assert(2 * kLeafW == 64, "one move per lane");
  const int lane = t & 63;
  const int my_src = mv_src[lane < moves ? lane : moves - 1];
  const int my_dst = mv_dst[lane < moves ? lane : moves - 1];
  const int i = blockIdx.x * blockDim.x + t;
  const bool act = i < ncols;
  int c = col_lo + (act ? i : 0);
  if (c >= skip_lo) c += skip_w;
  T vals[2 * kLeafW];
#pragma unroll
  for (int e = 0; e < 2 * kLeafW; e++) {
    // unconditional loads (a clamped, valid row) so all are in flight together
    vals[e] = A[(int64_t)__builtin_amdgcn_readlane(my_src, e) * lda + c];
  }
#pragma unroll
  for (int e = 0; e < 2 * kLeafW; e++)
    if (act && e < moves) A[(int64_t)__builtin_amdgcn_readlane(my_dst, e) * lda + c] = vals[e];
}

// Replay interchanges k1..k2-1 (in order) over the columns [col_lo, col_hi)
// minus [skip_lo, skip_hi): laswp / laswp_matrix (panel.mojo:1824-1852,
// :2279-2313), one thread per column.
template <typename T>
__global__ void laswp_kernel(T* __restrict__ A, int lda, int col_lo, int ncols, int skip_lo, int skip_w,
                             const int32_t* __restrict__ ipiv, int k1, int k2) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncols) return;
  int c = col_lo + i;
  if (c >= skip_lo) c += skip_w;
  for (int j = k1; j < k2; j++) {
    int o = ipiv[j];
    if (o != j) {
      T a = A[(int64_t)j * lda + c];
      T b = A[(int64_t)o * lda + c];
      A[(int64_t)j * lda + c] = b;
      A[(int64_t)o * lda + c] = a;
    }
  }
}

// Net permutation of the interchange sequence ipiv[0..n): row i of the
// permuted matrix is row perm[i] of the original one, which is what laswp
// over all n pivots (panel.mojo:1824-1852) leaves behind.  The sequence is a
// dependent chain, so one thread replays it on an identity vector; in LDS a
// step costs a few dozen cycles instead of the two dependent global
// round trips of a swap in place.  Pivot values are clamped to [0, n), so a
// corrupt ipiv yields a wrong permutation but no out-of-range access.
// The same permutation with the swaps taken 64 at a time.  A chunk's 64
// swaps, applied in order, permute at most 128 positions: its own 64 and up
// to 64 targets below it (ipiv[i] >= i).  A wavefront replays the chunk on
// labels -- slot s holds position pos_s and, after each swap, which
// position's value sits there (cont_s) -- so the chunk's net effect is
// perm'[pos_s] = perm[cont_s] for every touched slot: all reads, then all
// writes.  Sixteen wavefronts work out sixteen chunks at a time into LDS;
// wavefront 0 then applies them in order to the permutation held in LDS.
constexpr int kPermBatch = 16;  // chunks per round (one per wavefront)
__global__ void __launch_bounds__(1024) perm_chunks_kernel(int n, const int32_t* __restrict__ ipiv,
                                                           int32_t* __restrict__ perm) {
  extern __shared__ int s[];  // the permutation, n entries
  __shared__ int mdst[kPermBatch * 128], msrc[kPermBatch * 128], mcnt[kPermBatch];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  for (int i = t; i < n; i += blockDim.x) s[i] = i;
  const int nchunks = (n + 63) / 64;
  for (int c0 = 0; c0 < nchunks; c0 += kPermBatch) {
    const int c = c0 + wv;
    if (wv < kPermBatch && c < nchunks) {
      const int p0 = 64 * c, m = min(64, n - p0);
      const int iv = lane < m ? min(max(ipiv[p0 + lane], 0), n - 1) : p0 + lane;
      int pos0 = p0 + lane, cont0 = pos0;  // slot lane: position p0 + lane
      int pos1 = -1, cont1 = -1;           // slot 64 + lane: a target outside the chunk
      int nhi = 0;
      for (int j = 0; j < m; j++) {
        const int q = __builtin_amdgcn_readlane(iv, j);
        if (q == p0 + j) continue;
        int tq;
        if (q >= p0 && q < p0 + 64) {
          tq = q - p0;
        } else {
          const unsigned long long hit = __ballot(lane < nhi && pos1 == q);
          if (hit) {
            tq = 64 + __ffsll((long long)hit) - 1;
          } else {
            tq = 64 + nhi;
            if (lane == nhi) {
              pos1 = q;
              cont1 = q;
            }
            nhi++;
          }
        }
        const int a = __builtin_amdgcn_readlane(cont0, j);
        const int b = tq < 64 ? __builtin_amdgcn_readlane(cont0, tq) : __builtin_amdgcn_readlane(cont1, tq - 64);
        if (lane == j) cont0 = b;
        if (tq < 64) {
          if (lane == tq) cont0 = a;
        } else if (lane == tq - 64) {
          cont1 = a;
        }
      }
      // compact the moved slots
      const bool mv0 = cont0 != pos0, mv1 = lane < nhi && cont1 != pos1;
      const unsigned long long b0 = __ballot(mv0), b1 = __ballot(mv1);
      const int base1 = __popcll(b0);
      int* d = mdst + wv * 128;
      int* sr = msrc + wv * 128;
      if (mv0) {
        const int at = __popcll(b0 & ((1ull << lane) - 1ull));
        d[at] = pos0;
        sr[at] = cont0;
      }
      if (mv1) {
        const int at = base1 + __popcll(b1 & ((1ull << lane) - 1ull));
        d[at] = pos1;
        sr[at] = cont1;
      }
      if (lane == 0) mcnt[wv] = base1 + __popcll(b1);
    }
    __syncthreads();  // this round's moves, and (first round) the identity, are in LDS
    if (wv == 0) {
      for (int cc = 0; cc < kPermBatch && c0 + cc < nchunks; cc++) {
        const int cnt = mcnt[cc];
        const int* d = mdst + cc * 128;
        const int* sr = msrc + cc * 128;
        const int v0 = lane < cnt ? s[sr[lane]] : 0;
        const int v1 = lane + 64 < cnt ? s[sr[lane + 64]] : 0;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // every read before any write
        if (lane < cnt) s[d[lane]] = v0;
        if (lane + 64 < cnt) s[d[lane + 64]] = v1;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      }
    }
    __syncthreads();  // the moves' LDS is free for the next round
  }
  for (int i = t; i < n; i += blockDim.x) perm[i] = s[i];
}

template <int IN_LDS>
__global__ void __launch_bounds__(1024) perm_kernel(int n, const int32_t* __restrict__ ipiv,
                                                     int32_t* __restrict__ perm) {
  extern __shared__ int s_perm[];
  int* s = IN_LDS ? s_perm : perm;
  const int t = threadIdx.x;
  for (int i = t; i < n; i += blockDim.x) s[i] = i;
  __syncthreads();
  if (t == 0) {
    const auto rs = buf_rsrc(ipiv);
    for (int j0 = 0; j0 < n; j0 += 16) {
      int q[16];
#pragma unroll
      for (int u = 0; u < 16; u++)
        q[u] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, j0 + u < n ? 4u * (uint32_t)(j0 + u) : kBufOob, 0, 0);
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const int j = j0 + u;
        if (j < n) {
          const int p = min(max(q[u], 0), n - 1);
          const int a = s[j], b = s[p];
          s[j] = b;
          s[p] = a;
        }
      }
    }
  }
  __syncthreads();
  if (IN_LDS)
    for (int i = t; i < n; i += blockDim.x) perm[i] = s[i];
}

// out[i][c] = in[perm[i]][c] for c < ncols, converting Ti to To.
template <typename Ti, typename To>
__global__ void __launch_bounds__(256) gather_rows_kernel(int n, int ncols, const int32_t* __restrict__ perm,
                                                          const Ti* __restrict__ in, int ldi, To* __restrict__ out,
                                                          int ldo) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * ncols) return;
  const int i = (int)(idx / ncols), c = (int)(idx % ncols);
  out[(int64_t)i * ldo + c] = (To)in[(int64_t)perm[i] * ldi + c];
}

template <typename T>
__global__ void diag_kernel(int n, const T* __restrict__ A, int lda, T* __restrict__ d) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = A[(int64_t)i * lda + i];
}

template <typename T>
__global__ void tril_kernel(int n, T* __restrict__ A, int lda) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * n) return;
  int i = (int)(idx / n), c = (int)(idx % n);
  if (c > i) A[(int64_t)i * lda + c] = T(0);
}

__global__ void zero_i32(int32_t* p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Recursive triangular solve: split op(T) in two, solve one diagonal block,
// update the other half of the right-hand sides with the MFMA GEMM, solve the
// other block.  VEC_ROWS = 0: the vectors are B's columns (B is n x nvec);
// VEC_ROWS = 1: they are B's rows (B is nvec x n).
template <typename T, int VEC_ROWS>
int trsm_rec(nmx_ctx* ctx, int upper, int unit, int trans, int n, int nvec, const T* Tm, int ldt, T* B, int ldb) {
  if (n <= 0 || nvec <= 0) return NMX_OK;
  // a strip's offsets are 32-bit: rows of an operand more than 2 GiB apart
  // (hundreds of thousands of columns) go through in lower strips
  const int64_t span = (VEC_ROWS ? 32 : (int64_t)n) * ldb, tspan = (int64_t)n * ldt;
  const bool fits = std::max(span, tspan) * (int64_t)sizeof(T) < 0x7FFFFFFF;
  if (n <= kStripMax && (fits || n <= 16))
    return trsm_strip<T>(ctx, upper, unit, trans, VEC_ROWS, n, nvec, Tm, ldt, B, ldb);
  const int n1 = n > 64 ? trsm_split(n) : ((n / 2 + 15) / 16) * 16;
  const int n2 = n - n1;
  const T* T11 = Tm;
  const T* T22 = Tm + (int64_t)n1 * ldt + n1;
  const T* Tlo = Tm + (int64_t)n1 * ldt;  // stored rows n1.., cols 0..n1
  const T* Tup = Tm + n1;                 // stored rows 0..n1, cols n1..
  // vector halves
  T* B1 = B;
  T* B2 = VEC_ROWS ? B + n1 : B + (int64_t)n1 * ldb;
  // op(T)21 (forward) or op(T)12 (backward) as stored block + transpose flag
  if (!upper) {
    NMX_TRY((trsm_rec<T, VEC_ROWS>(ctx, upper, unit, trans, n1, nvec, T11, ldt, B1, ldb)));
    // op(T)21 = trans ? (T12)^T : T21
    const T* blk = trans ? Tup : Tlo;
    if (!VEC_ROWS) {
      NMX_TRY(gemm_launch<T>(ctx, trans, 0, n2, nvec, n1, T(-1), blk, ldt, B1, ldb, T(1), B2, ldb, 0));
    } else {
      // rows: X2 -= X1 op(T)21^T
      NMX_TRY(gemm_launch<T>(ctx, 0, trans ? 0 : 1, nvec, n2, n1, T(-1), B1, ldb, blk, ldt, T(1), B2, ldb, 0));
    }
    NMX_TRY((trsm_rec<T, VEC_ROWS>(ctx, upper, unit, trans, n2, nvec, T22, ldt, B2, ldb)));
  } else {
    NMX_TRY((trsm_rec<T, VEC_ROWS>(ctx, upper, unit, trans, n2, nvec, T22, ldt, B2, ldb)));
    // op(T)12 = trans ? (T21)^T : T12
    const T* blk = trans ? Tlo : Tup;
    if (!VEC_ROWS) {
      NMX_TRY(gemm_launch<T>(ctx, trans, 0, n1, nvec, n2, T(-1), blk, ldt, B2, ldb, T(1), B1, ldb, 0));
    } else {
      NMX_TRY(gemm_launch<T>(ctx, 0, trans ? 0 : 1, nvec, n1, n2, T(-1), B2, ldb, blk, ldt, T(1), B1, ldb, 0));
    }
    NMX_TRY((trsm_rec<T, VEC_ROWS>(ctx, upper, unit, trans, n1, nvec, T11, ldt, B1, ldb)));
  }
  return NMX_OK;
}

}  // namespace

template <typename T>
int trsm_left(nmx_ctx* ctx, int upper, int unit, int trans, int n, int nrhs, const T* Tm, int ldt, T* B, int ldb) {
  return trsm_rec<T, 0>(ctx, upper, unit, trans, n, nrhs, Tm, ldt, B, ldb);
}

template <typename T>
int trsm_right_lower_t(nmx_ctx* ctx, int m, int n, const T* L, int ldl, T* X, int ldx) {
  // X := X L^-T  <=>  each row x of X solves L x^T = x^T (forward, non-unit)
  return trsm_rec<T, 1>(ctx, 0, 0, 0, n, m, L, ldl, X, ldx);
}

// X := X U^-1 with U upper n x n (rows of X solve U^T x^T = a^T).
int trsm_rec_rows_upper(nmx_ctx* ctx, int m, int n, const float* U, int ldu, float* X, int ldx) {
  return trsm_rec<float, 1>(ctx, 0, 0, 1, n, m, U, ldu, X, ldx);
}

template <typename T>
int laswp_launch(nmx_ctx* ctx, T* A, int lda, int col_lo, int col_hi, int skip_lo, int skip_hi, const int32_t* ipiv,
                 int k1, int k2) {
  if (k2 <= k1 || col_hi <= col_lo) return NMX_OK;
  int s_lo = skip_lo < col_lo ? col_lo : skip_lo;
  int s_hi = skip_hi > col_hi ? col_hi : skip_hi;
  int skip_w = s_hi > s_lo ? s_hi - s_lo : 0;
  if (skip_w == 0) s_lo = col_hi;
  int ncols = col_hi - col_lo - skip_w;
  if (ncols <= 0) return NMX_OK;
  ProfScope ps(ctx, K_LASWP, 0.0, 4.0 * sizeof(T) * (double)ncols * (k2 - k1));
  if (k2 - k1 <= kLeafW)
    laswp_gather_kernel<T><<<ceil_div(ncols, 256), 256, 0, ctx->stream>>>(A, lda, col_lo, ncols, s_lo, skip_w, ipiv, k1,
                                                                           k2);
  else
    laswp_kernel<T><<<ceil_div(ncols, 256), 256, 0, ctx->stream>>>(A, lda, col_lo, ncols, s_lo, skip_w, ipiv, k1, k2);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

int perm_from_ipiv(nmx_ctx* ctx, int n, const int32_t* ipiv, int32_t* perm) {
  if (n <= 0) return NMX_OK;
  ProfScope ps(ctx, K_LASWP, 0.0, 8.0 * n);
  const size_t lds = sizeof(int32_t) * (size_t)n;
  if (lds <= kPermLdsBytes)
    perm_chunks_kernel<<<1, 1024, lds, ctx->stream>>>(n, ipiv, perm);
  else
    perm_kernel<0><<<1, 1024, 0, ctx->stream>>>(n, ipiv, perm);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

template <typename Ti, typename To>
int gather_rows(nmx_ctx* ctx, int n, int ncols, const int32_t* perm, const Ti* in, int ldi, To* out, int ldo) {
  const int64_t total = (int64_t)n * ncols;
  if (total <= 0) return NMX_OK;
  ProfScope ps(ctx, K_LASWP, 0.0, (double)total * (sizeof(Ti) + sizeof(To)) + 4.0 * n);
  gather_rows_kernel<Ti, To><<<(unsigned)((total + 255) / 256), 256, 0, ctx->stream>>>(n, ncols, perm, in, ldi, out,
                                                                                       ldo);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}
template int gather_rows<double, double>(nmx_ctx*, int, int, const int32_t*, const double*, int, double*, int);
template int gather_rows<float, float>(nmx_ctx*, int, int, const int32_t*, const float*, int, float*, int);
template int gather_rows<double, float>(nmx_ctx*, int, int, const int32_t*, const double*, int, float*, int);

template <typename T>
int getf2_leaf_launch(nmx_ctx* ctx, int n, T* A, int lda, int r0, int c0, int w, int32_t* ipiv, int32_t* info,
                      int swap_others) {
  const int m = n - r0;
  if (m <= 0 || w <= 0) return NMX_OK;
  if (w > kLeafW) return NMX_ERR_UNSUPPORTED;
  // one row per thread while the panel fits 32 workgroups of 512 rows, two
  // above that
  const bool one_row = m <= kLeafT * kMaxParts;
  const int parts = m <= kLeafMaxT ? 1 : ceil_div(m, one_row ? kLeafT : kLeafT * 2);
  if (parts > kMaxParts) return NMX_ERR_UNSUPPORTED;  // n - r0 <= kLeafMaxRows
  uint32_t epoch0 = 0;
  NMX_TRY(nmx_epoch_reserve(ctx, (uint32_t)w, &epoch0));
  uint64_t* mb = (uint64_t*)ctx->mailbox;
  int* err = ctx->err;
  {
    ProfScope ps(ctx, K_LEAF, (double)m * w * w, 2.0 * sizeof(T) * (double)m * w);
    // At most 8 x 32 workgroups of 512 threads: one per CU of an otherwise
    // idle device (the stream orders this launch after the previous kernel).
    // A participant that is not resident makes the others' bounded waits
    // expire, which the context reports as NMX_ERR_SYNC_TIMEOUT.
    const int grid = parts == 1 ? 1 : parts * kXcds;
    // in one workgroup: only the wavefronts that hold rows.  Up to 1024 rows
    // that is faster than an exchange between two (2.8 us a column)
    const int threads = parts == 1 ? ceil_div(m, 64) * 64 : kLeafT;
    if (parts == 1)
      getf2_leaf<T, 1, false><<<grid, threads, 0, ctx->stream>>>(A, lda, n, r0, c0, w, ipiv, info, mb, epoch0, parts, err);
    else if (one_row)
      getf2_leaf<T, 1, true><<<grid, kLeafT, 0, ctx->stream>>>(A, lda, n, r0, c0, w, ipiv, info, mb, epoch0, parts, err);
    else
      getf2_leaf<T, 2, true><<<grid, kLeafT, 0, ctx->stream>>>(A, lda, n, r0, c0, w, ipiv, info, mb, epoch0, parts, err);
    NMX_HIP(ctx, hipGetLastError());
  }
  if (swap_others) return laswp_launch<T>(ctx, A, lda, 0, n, c0, c0 + w, ipiv, r0, r0 + w);
  return NMX_OK;
}

template <typename T>
int diag_launch(nmx_ctx* ctx, int n, const T* A, int lda, T* d) {
  if (n <= 0) return NMX_OK;
  diag_kernel<T><<<ceil_div(n, 256), 256, 0, ctx->stream>>>(n, A, lda, d);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

int zero_info(nmx_ctx* ctx, int32_t* info) {
  zero_i32<<<1, 64, 0, ctx->stream>>>(info, 1);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

template <typename T>
int tril_launch(nmx_ctx* ctx, int n, T* A, int lda) {
  int64_t total = (int64_t)n * n;
  if (total <= 0) return NMX_OK;
  tril_kernel<T><<<(unsigned)((total + 255) / 256), 256, 0, ctx->stream>>>(n, A, lda);
  NMX_HIP(ctx, hipGetLastError());
  return NMX_OK;
}

#define INST(T)                                                                                                     \
  template int trsm_left<T>(nmx_ctx*, int, int, int, int, int, const T*, int, T*, int);                            \
  template int trsm_right_lower_t<T>(nmx_ctx*, int, int, const T*, int, T*, int);                                  \
  template int laswp_launch<T>(nmx_ctx*, T*, int, int, int, int, int, const int32_t*, int, int);                   \
  template int getf2_leaf_launch<T>(nmx_ctx*, int, T*, int, int, int, int, int32_t*, int32_t*, int);               \
  template int diag_launch<T>(nmx_ctx*, int, const T*, int, T*);                                                   \
  template int tril_launch<T>(nmx_ctx*, int, T*, int);
INST(double)
INST(float)
