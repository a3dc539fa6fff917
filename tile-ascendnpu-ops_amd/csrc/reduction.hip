// Reductions for gfx950: LogSumExp and Argmax / Argmin over the last dimension
// of a row-major [M, N] tensor, over the middle dimension of [outer, N, inner]
// (column kernel, below) or over the outer two of [R, M, L].
//
// Rows.  A wavefront streams its share of a row in 16-byte packs, U packs per
// lane in flight, folds them into a per-lane partial, and the 64 partials meet
// in a shuffle butterfly.  What bounds the kernel is HBM where the rows fill
// the chip, and the latency of one wavefront's chain of loads where they do
// not, so the number of wavefronts per row follows the row count (plan_rows):
// 1 (four rows per workgroup), 4, 16 (a 1024-thread workgroup), or several
// 4-wavefront workgroups per row whose partials a second launch merges.
#include <algorithm>

#include <float.h>

#include "common.h"

namespace tileops {

constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------------------
// LogSumExp: online (max, scaled-sum) per lane.
//
// m is the running max of everything folded so far (NaN never wins the
// compare, so m stays in [-inf, +inf]); s = sum exp(x - shift(m)) where
// shift(m) = m for a finite max and 0 for an infinite one, as torch does.
// That reproduces torch.logsumexp's special cases and keeps every finite
// max up to FLT_MAX finite:
//   all -inf    -> shift 0, s = 0, log 0 + 0 = -inf
//   any +inf    -> shift 0, exp(+inf) = +inf in s   (result +inf)
//   any NaN     -> NaN enters s                     (result NaN)
// s == 0 exactly when m == -inf (a finite max contributes exp(0) = 1), and
// such a sum is rescaled to 0 without evaluating a factor that could be
// exp(+huge) = inf (0 * inf would be NaN).
// ---------------------------------------------------------------------------
struct LseState {
  float m;  // running max, -inf while nothing finite or +inf was folded
  float s;  // sum of exp(x - lse_shift(m))
};

__device__ __forceinline__ float lse_shift(float m) {
  return __builtin_fabsf(m) <= FLT_MAX ? m : 0.0f;
}

// s, taken relative to shift `from`, re-expressed relative to shift `to`.
__device__ __forceinline__ float lse_rescale(float s, float from, float to) {
  const float f = __builtin_amdgcn_exp2f((from - to) * kLog2e);
  return s == 0.0f ? 0.0f : s * f;
}

__device__ __forceinline__ LseState lse_merge(LseState a, LseState b) {
  const float m = a.m > b.m ? a.m : b.m;
  const float sh = lse_shift(m);
  return {m, lse_rescale(a.s, lse_shift(a.m), sh) + lse_rescale(b.s, lse_shift(b.m), sh)};
}

template <int CNT>
__device__ __forceinline__ void lse_fold(LseState& st, const float (&v)[CNT]) {
  float bm = v[0];
#pragma unroll
  for (int i = 1; i < CNT; ++i) bm = v[i] > bm ? v[i] : bm;
  const float mn = bm > st.m ? bm : st.m;
  const float sh = lse_shift(mn);
  // exp(x - m) as exp2((x - m) * log2 e): subtracting first keeps the
  // exponent exact for large |m| (an fma(x, log2 e, -m log2 e) would leave
  // the rounding residue of m log2 e, ~1e31 at |m| ~ 1e38).
  float acc = lse_rescale(st.s, lse_shift(st.m), sh);
#pragma unroll
  for (int i = 0; i < CNT; ++i) acc += __builtin_amdgcn_exp2f((v[i] - sh) * kLog2e);
  st.m = mn;
  st.s = acc;
}

// Merged over aligned groups of G lanes.
template <int G>
__device__ __forceinline__ LseState lse_wave(LseState st) {
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) {
    LseState other{__shfl_xor(st.m, o, 64), __shfl_xor(st.s, o, 64)};
    st = lse_merge(st, other);
  }
  return st;
}

__device__ __forceinline__ float lse_final(LseState st) {
  // log(s) + shift; s >= 1 whenever the max is finite.
  return logf(st.s) + lse_shift(st.m);
}

// ---------------------------------------------------------------------------
// Arg-reduction (value, index) with torch.argmax semantics: NaN beats every
// number, equal values keep the lowest index.  Index -1 marks "no element".
// ---------------------------------------------------------------------------
struct ArgState {
  float v;
  int i;
};

template <bool IS_MIN>
__device__ __forceinline__ bool arg_better(float a, int ia, float b, int ib) {
  if (ia < 0) return false;
  if (ib < 0) return true;
  const bool an = a != a, bn = b != b;
  if (an || bn) return an && (!bn || ia < ib);
  if (a == b) return ia < ib;
  return IS_MIN ? a < b : a > b;
}

// In-lane update where `i` is known to exceed every index already folded:
// replace unless the current best is NaN, or `a` does not strictly beat it
// (a NaN `a` beats any number).
template <bool IS_MIN>
__device__ __forceinline__ void arg_step(ArgState& st, float a, int i) {
  const bool take = (st.i < 0) | ((st.v == st.v) & (IS_MIN ? !(a >= st.v) : !(a <= st.v)));
  st.v = take ? a : st.v;
  st.i = take ? i : st.i;
}

template <bool IS_MIN, int G>
__device__ __forceinline__ ArgState arg_wave(ArgState st) {
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) {
    ArgState other{__shfl_xor(st.v, o, 64), __shfl_xor(st.i, o, 64)};
    if (arg_better<IS_MIN>(other.v, other.i, st.v, st.i)) st = other;
  }
  return st;
}

// ---------------------------------------------------------------------------
// OP 0 = logsumexp, 1 = argmax, 2 = argmin.
// ---------------------------------------------------------------------------
template <int OP> struct RowState;
template <> struct RowState<0> { typedef LseState S; };
template <> struct RowState<1> { typedef ArgState S; };
template <> struct RowState<2> { typedef ArgState S; };

template <int OP>
__device__ __forceinline__ typename RowState<OP>::S row_init() {
  if constexpr (OP == 0) return LseState{-INFINITY, 0.0f};
  else return ArgState{0.0f, -1};
}

template <int OP>
__device__ __forceinline__ typename RowState<OP>::S row_merge(typename RowState<OP>::S a,
                                                              typename RowState<OP>::S b) {
  if constexpr (OP == 0) return lse_merge(a, b);
  else return arg_better<OP == 2>(b.v, b.i, a.v, a.i) ? b : a;
}

template <int OP, int G = 64>
__device__ __forceinline__ typename RowState<OP>::S row_wave(typename RowState<OP>::S st) {
  if constexpr (OP == 0) return lse_wave<G>(st);
  else return arg_wave<OP == 2, G>(st);
}

template <typename T, int OP>
__device__ __forceinline__ void row_store(void* out, int64_t row, typename RowState<OP>::S st) {
  if constexpr (OP == 0) static_cast<T*>(out)[row] = Elem<T>::from_f32(lse_final(st));
  else static_cast<int64_t*>(out)[row] = st.i < 0 ? 0 : (int64_t)st.i;
}

// WPR wavefronts of one workgroup share a row, and `nsplit` workgroups; a
// wavefront takes every (WPR * nsplit)-th chunk of 64 packs, U of them in
// flight per step.  ALIGNED: every row starts on a 16-byte boundary and holds
// whole packs.  Otherwise the row's packs start at its first aligned element;
// the row's first wavefront folds the elements before them in its first step
// and those after them in its last, one per lane,
// so that an odd row length costs no more loads than an even one (LogSumExp
// bf16 16384 x 4097: 73.9 us with one element per lane and load, 28.9 so).
// PARTS: `out` holds partials, `per` for each of the `keep` outputs, of which
// rows r, r + keep, .. give nsplit each; else nsplit is 1 (as a parameter its
// divisions and products cost every row: Argmax fp32 100000 x 500 44.2 us and
// 41.7).  All U loads of a step are issued before their uses, past-the-end ones
// clamped onto the row's last pack: a load under a branch of its own was waited
// for there (then, us: that shape 36.9, Argmax bf16 32768 x 4096 61.5 -> 42.2,
// 1024 x 32768 18.4 -> 12.9; LogSumExp bf16 32768 x 4096 48.7 -> 43.1, 700 x
// 16384 8.5 -> 6.2).
struct PartMap {
  int64_t keep;
  int per;
};
template <typename T, int OP, int WPR, int U, bool ALIGNED, bool PARTS>
__global__ __launch_bounds__(WPR > 4 ? 64 * WPR : 256) void row_reduce_kernel(
    const T* __restrict__ x, void* __restrict__ out, int64_t M, int64_t N, int nstep, int splits,
    PartMap pm) {
  typedef typename RowState<OP>::S S;
  constexpr int V = Elem<T>::kVec;
  constexpr int WPB = WPR > 4 ? WPR : 4;  // wavefronts per workgroup
  constexpr int ROWS_PER_BLOCK = WPB / WPR;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_in_row = wave % WPR;
  const int nsplit = PARTS ? splits : 1;
  const int64_t ngroup = (M + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK * nsplit;

  __shared__ S part[WPB];

  for (int64_t group = blockIdx.x; group < ngroup; group += gridDim.x) {
    const int split = nsplit == 1 ? 0 : (int)(group % nsplit);
    const int64_t row = (nsplit == 1 ? group : group / nsplit) * ROWS_PER_BLOCK + wave / WPR;
    S st = row_init<OP>();
    if (row < M) {
      const T* xr = x + row * N;
      int head = 0;
      if constexpr (!ALIGNED) {
        const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(xr) & 15u);
        head = (int)min((int64_t)((16u - mis) & 15u) / (int64_t)sizeof(T), N);
      }
      const int np = (int)((N - head) / V);  // at least 64: shorter rows are short_row_kernel's
      const T* xb = xr + head;
      const int gw = split * WPR + wave_in_row, nw = nsplit * WPR;
      // what a slot past the row reads as: exp(-inf) adds 0 to a sum, and the
      // worst value with an index past every other never wins
      constexpr float kPast = OP == 2 ? INFINITY : -INFINITY;
      for (int k = 0; k < nstep; ++k) {
        constexpr int EDGE = ALIGNED ? 0 : 2;
        float vals[U * V + EDGE];
        const int c0 = (k * U * nw + gw) * 64;
        if (c0 >= np && gw > 0) break;  // the first wavefront has the row's end to fold
        Pack<T> p[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          p[u] = load_pack_nt(xb + (int64_t)min(c0 + u * nw * 64 + lane, np - 1) * V);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int e = 0; e < V; ++e) vals[u * V + e] = Elem<T>::to_f32(p[u].v[e]);
        }
        if (c0 + ((U - 1) * nw + 1) * 64 > np) {  // the row ends in this step
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const bool in = c0 + u * nw * 64 + lane < np;
#pragma unroll
            for (int e = 0; e < V; ++e) vals[u * V + e] = in ? vals[u * V + e] : kPast;
          }
        }
        bool first = false, last = false;
        const int64_t t = head + (int64_t)np * V + lane;
        if constexpr (!ALIGNED) {
          first = gw == 0 && k == 0 && lane < head;
          last = gw == 0 && k == nstep - 1 && t < N;
          vals[U * V] = vals[U * V + 1] = -INFINITY;
          if (first) vals[U * V] = Elem<T>::to_f32(xr[lane]);
          if (last) vals[U * V + 1] = Elem<T>::to_f32(xr[t]);
        }
        if constexpr (OP == 0) {
          lse_fold<U * V + EDGE>(st, vals);
        } else {
          if constexpr (!ALIGNED) {
            if (first) arg_step<OP == 2>(st, vals[U * V], lane);
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t i0 = (uint32_t)head + (uint32_t)(c0 + u * nw * 64 + lane) * V;
#pragma unroll
            for (int e = 0; e < V; ++e) arg_step<OP == 2>(st, vals[u * V + e], (int)(i0 + e));
          }
          if constexpr (!ALIGNED) {
            if (last) arg_step<OP == 2>(st, vals[U * V + 1], (int)t);
          }
        }
      }
    }
    st = row_wave<OP>(st);
    if constexpr (WPR > 1) {
      if (lane == 0) part[wave] = st;
      __syncthreads();
      if constexpr (WPR > 4) {
        if (wave == 0) st = row_wave<OP, WPR>(part[lane % WPR]);
      } else {
        if (wave == 0) {
          st = part[0];
#pragma unroll
          for (int w = 1; w < WPR; ++w) st = row_merge<OP>(st, part[w]);
        }
      }
      __syncthreads();
    }
    if (lane == 0 && wave_in_row == 0 && row < M) {
      if constexpr (PARTS)
        static_cast<S*>(out)[row % pm.keep * pm.per + row / pm.keep * nsplit + split] = st;
      else
        row_store<T, OP>(out, row, st);
    }
  }
}

// Short rows: G lanes per row, one load per lane, 64 / G rows per wavefront, so
// that a row costs log2 G merges instead of six and no lane group idles (one
// wavefront per row and this, us: Argmax fp16 524288 x 4: 120 -> 6.8,
// LogSumExp bf16 88000 x 128: 50 -> 8.9).  PACKS: a lane takes one pack;
// ragged rows as in row_reduce_kernel (G >= 16 lanes hold the elements before
// and after the packs).  Otherwise a lane takes one element.
template <typename T, int OP, int G, bool PACKS, bool ALIGNED, bool PARTS>
__global__ __launch_bounds__(256) void short_row_kernel(const T* __restrict__ x,
                                                        void* __restrict__ out, int64_t M, int N,
                                                        PartMap pm, int64_t block0) {
  constexpr int V = PACKS ? Elem<T>::kVec : 1, EDGE = PACKS && !ALIGNED ? 2 : 0;
  static_assert(EDGE == 0 || G >= Elem<T>::kVec, "a lane per edge element");
  const int64_t row = (block0 + blockIdx.x) * (256 / G) + threadIdx.x / G;
  const int lane = threadIdx.x % G;
  typename RowState<OP>::S st = row_init<OP>();
  if (row < M) {
    const T* xr = x + row * N;
    int head = 0;
    if constexpr (EDGE > 0) {
      const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(xr) & 15u);
      head = min((int)(((16u - mis) & 15u) / sizeof(T)), N);
    }
    const int np = (N - head) / V, t = head + np * V + lane;
    float vals[V + EDGE];
#pragma unroll
    for (int e = 0; e < V + EDGE; ++e) vals[e] = -INFINITY;
    if (lane < np) {
      if constexpr (PACKS) {
        const Pack<T> p = load_pack_nt(xr + head + lane * V);
#pragma unroll
        for (int e = 0; e < V; ++e) vals[e] = Elem<T>::to_f32(p.v[e]);
      } else {
        vals[0] = Elem<T>::to_f32(xr[lane]);
      }
    }
    if constexpr (EDGE > 0) {
      if (lane < head) vals[V] = Elem<T>::to_f32(xr[lane]);
      if (t < N) vals[V + 1] = Elem<T>::to_f32(xr[t]);
    }
    if constexpr (OP == 0) {
      lse_fold<V + EDGE>(st, vals);
    } else {
      if constexpr (EDGE > 0) {
        if (lane < head) arg_step<OP == 2>(st, vals[V], lane);
      }
      if (lane < np) {
#pragma unroll
        for (int e = 0; e < V; ++e) arg_step<OP == 2>(st, vals[e], head + lane * V + e);
      }
      if constexpr (EDGE > 0) {
        if (t < N) arg_step<OP == 2>(st, vals[V + 1], t);
      }
    }
  }
  st = row_wave<OP, G>(st);
  if (row < M && lane == 0) {
    if constexpr (PARTS)
      static_cast<typename RowState<OP>::S*>(out)[row % pm.keep * pm.per + row / pm.keep] = st;
    else
      row_store<T, OP>(out, row, st);
  }
}

// The nsplit partials of each output, one wavefront per output.
template <typename T, int OP>
__global__ __launch_bounds__(256) void merge_partials_kernel(
    const typename RowState<OP>::S* __restrict__ part, void* __restrict__ out, int64_t M,
    int nsplit, int64_t block0) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (block0 + blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  typename RowState<OP>::S st = row_init<OP>();
  for (int i = lane; i < nsplit; i += 64) st = row_merge<OP>(st, part[row * nsplit + i]);
  st = row_wave<OP>(st);
  if (lane == 0) row_store<T, OP>(out, row, st);
}

template <typename T, int OP>
static int launch_merge(const void* ws, void* out, int64_t M, int nsplit, hipStream_t s) {
  return launch_slices((M + 3) / 4, 256, [&](int64_t block0, dim3 grid) {
    merge_partials_kernel<T, OP><<<grid, dim3(256), 0, s>>>(
        static_cast<const typename RowState<OP>::S*>(ws), out, M, nsplit, block0);
  });
}

// How a [M, N] row reduction is laid out.  One wavefront per row from 3072
// rows up (a dozen wavefronts per CU; LogSumExp bf16 3072 x 4096 7.9 us, 9.3 with
// four), four below, sixteen where at most 512 rows leave each of those work
// (512 x 32768: LogSumExp bf16 9.9 us with four and 9.6 with sixteen, Argmax 11.4
// and 10.3; 1024 rows: 14.9 and 16.6; 512 x 8192: 5.5 and 8.4).  At most 128 rows
// (two CUs each) of 256 chunks or more (sixteen wavefronts would take four steps
// and more, ~2 us each) are split over workgroups of four wavefronts, one step
// each up to 1024 workgroups; the merge launch and its scratch cost ~2.5 us on
// the GPU and ~4 us of an eager call's host time, so shorter rows stay whole
// (LogSumExp bf16 4 x 102400: 15.3 us with four wavefronts per row, 9.4 with
// sixteen, 6.3 split, but 10.4 and ~14 us per eager call; 4 x 131072 10.0 whole
// and 6.1 split; Argmax of 2^21 fp16 elements 143 with sixteen, 9.1 split, of
// 2^25 fp32 33.7 split).
// A wavefront keeps 4 packs per lane in flight, fewer where its whole share of
// the row is less (slots past the row still cost their exponentials).
struct RowPlan {
  int wpr, u, nsplit, nstep;
};
static RowPlan plan_rows(int64_t M, int64_t N, int vec, bool split = true) {
  const int64_t chunks = std::max<int64_t>((N / vec + 63) / 64, 1);
  RowPlan p{4, 4, 1, 0};
  if (M >= 256 * 12) p.wpr = 1;
  else if (M <= 512 && chunks >= 16 * 4) p.wpr = 16;
  if (split && M <= 128 && chunks >= 16 * 16) {
    p.wpr = 4;
    p.nsplit = (int)std::min<int64_t>((chunks + 15) / 16, 1024 / M);
  }
  if (p.wpr <= 4 && p.nsplit == 1) p.u = (int)std::min<int64_t>((chunks + p.wpr - 1) / p.wpr, 4);
  const int64_t per_step = (int64_t)p.u * p.wpr * p.nsplit;
  p.nstep = (int)((chunks + per_step - 1) / per_step);
  return p;
}

template <typename T, int OP, int WPR, int U, bool PARTS>
static void launch_rows(const T* x, void* out, int64_t M, int64_t N, const RowPlan& p,
                        PartMap pm, hipStream_t s) {
  const bool aligned = host_aligned16(x) && (N % Elem<T>::kVec) == 0;
  const int rows_per_block = WPR > 4 ? 1 : 4 / WPR;
  const int64_t blocks = (M + rows_per_block - 1) / rows_per_block * p.nsplit;
  const dim3 grid((unsigned)std::min<int64_t>(blocks, 256 * 32)), block(WPR > 4 ? 64 * WPR : 256);
  if (aligned)
    row_reduce_kernel<T, OP, WPR, U, true, PARTS><<<grid, block, 0, s>>>(x, out, M, N, p.nstep, p.nsplit, pm);
  else
    row_reduce_kernel<T, OP, WPR, U, false, PARTS><<<grid, block, 0, s>>>(x, out, M, N, p.nstep, p.nsplit, pm);
}

template <typename T, int OP, int WPR, bool PARTS>
static void launch_rows_u(const T* x, void* out, int64_t M, int64_t N, const RowPlan& p,
                          PartMap pm, hipStream_t s) {
  if (p.u == 1) launch_rows<T, OP, WPR, 1, PARTS>(x, out, M, N, p, pm, s);
  else if (p.u == 2) launch_rows<T, OP, WPR, 2, PARTS>(x, out, M, N, p, pm, s);
  else if (p.u == 3) launch_rows<T, OP, WPR, 3, PARTS>(x, out, M, N, p, pm, s);
  else launch_rows<T, OP, WPR, 4, PARTS>(x, out, M, N, p, pm, s);
}

template <typename T, int OP, bool PARTS>
static int launch_long(const T* x, void* out, int64_t M, int64_t N, const RowPlan& p, PartMap pm,
                       hipStream_t s) {
  if constexpr (PARTS && OP != 0)  // an index has partials of split rows alone (plan_rows)
    launch_rows<T, OP, 4, 4, true>(x, out, M, N, p, pm, s);
  else if (p.wpr == 1) launch_rows_u<T, OP, 1, PARTS>(x, out, M, N, p, pm, s);
  else if (p.wpr == 4) launch_rows_u<T, OP, 4, PARTS>(x, out, M, N, p, pm, s);
  else launch_rows<T, OP, 16, 4, PARTS>(x, out, M, N, p, pm, s);
  return launch_status();
}

// The short-row kernel takes rows of at most 64 packs; ragged rows of up to 16
// elements go element by element.
static bool short_rows(int64_t N, int vec) { return N / vec <= 64; }

template <typename T, int OP, bool PARTS>
static int launch_short(const T* x, void* out, int64_t M, int64_t N, PartMap pm, hipStream_t s) {
  constexpr int V = Elem<T>::kVec;
  const int n = (int)N, np = n / V;
  auto go = [&](auto kernel, int G) {
    const int64_t rows = 256 / G;
    return launch_slices((M + rows - 1) / rows, 256, [&](int64_t block0, dim3 grid) {
      kernel<<<grid, dim3(256), 0, s>>>(x, out, M, n, pm, block0);
    });
  };
  if (host_aligned16(x) && n % V == 0) {
    if (np <= 4) return go(short_row_kernel<T, OP, 4, true, true, PARTS>, 4);
    if (np <= 16) return go(short_row_kernel<T, OP, 16, true, true, PARTS>, 16);
    if (np <= 32) return go(short_row_kernel<T, OP, 32, true, true, PARTS>, 32);
    return go(short_row_kernel<T, OP, 64, true, true, PARTS>, 64);
  }
  if (n <= 4) return go(short_row_kernel<T, OP, 4, false, false, PARTS>, 4);
  if (n <= 16) return go(short_row_kernel<T, OP, 16, false, false, PARTS>, 16);
  if (np <= 16) return go(short_row_kernel<T, OP, 16, true, false, PARTS>, 16);
  if (np <= 32) return go(short_row_kernel<T, OP, 32, true, false, PARTS>, 32);
  return go(short_row_kernel<T, OP, 64, true, false, PARTS>, 64);
}

// Rows of x[M, N]; with keep > 0 rows r, r + keep, .. belong to output r
// (x[M / keep, keep, N] reduced over its outer two dimensions), merged from
// partials.
template <typename T, int OP>
static int launch_row_reduce(const void* xv, void* out, int64_t M, int64_t N, int64_t keep,
                             void* ws, size_t ws_bytes, hipStream_t s) {
  typedef typename RowState<OP>::S S;
  const T* x = static_cast<const T*>(xv);
  RowPlan p = plan_rows(M, N, Elem<T>::kVec);
  const int64_t folds = keep > 0 ? M / keep : 1, nout = M / folds;
  if (folds == 1 && p.nsplit > 1 && ws_bytes < (size_t)M * p.nsplit * sizeof(S))
    p = plan_rows(M, N, Elem<T>::kVec, false);  // no scratch
  PartMap pm{nout, 0};
  const bool is_short = short_rows(N, Elem<T>::kVec);
  if (folds > 1 || (p.nsplit > 1 && !is_short)) pm.per = (int)folds * (is_short ? 1 : p.nsplit);
  if (pm.per == 0)
    return is_short ? launch_short<T, OP, false>(x, out, M, N, pm, s)
                    : launch_long<T, OP, false>(x, out, M, N, p, pm, s);
  int e;
  if constexpr (OP == 0)
    e = is_short ? launch_short<T, OP, true>(x, ws, M, N, pm, s)
                 : launch_long<T, OP, true>(x, ws, M, N, p, pm, s);
  else
    e = launch_long<T, OP, true>(x, ws, M, N, p, pm, s);
  return e ? e : launch_merge<T, OP>(ws, out, nout, pm.per, s);
}

// ---------------------------------------------------------------------------
// Columns: x[outer, N, inner] reduced over N, read as it lies (the copy that
// moves the reduced dimension last costs a read and a write of the tensor, and
// short columns then made one wavefront per column: Argmax fp16 [4, 128, 4096]
// over dimension 0 126.6 us, 6.6 so).  A thread owns the V columns of one pack (one
// column where packs do not fit); TX threads cover neighbouring packs and 256
// / TX share a column's rows, U = 4 in flight each, and meet in LDS.  Bound by
// HBM where the columns fill the chip; `nsplit` workgroups share a column
// where they do not.
// ---------------------------------------------------------------------------
template <typename T, int OP, int V, int TX>
__global__ __launch_bounds__(256) void col_reduce_kernel(const T* __restrict__ x,
                                                         void* __restrict__ out, int64_t N,
                                                         int64_t inner, int64_t ntile, int nsplit,
                                                         int64_t block0) {
  typedef typename RowState<OP>::S S;
  constexpr int TY = 256 / TX, U = 4;
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int64_t block = block0 + blockIdx.x;
  const int64_t tile = block % ntile;
  const int64_t rest = block / ntile;
  const int split = (int)(rest % nsplit);
  const int64_t o = rest / nsplit;
  const int64_t c0 = (tile * TX + tx) * V;
  const int64_t per = (N + nsplit - 1) / nsplit;
  const int64_t n0 = split * per, n1 = min(N, n0 + per);

  S st[V];
#pragma unroll
  for (int e = 0; e < V; ++e) st[e] = row_init<OP>();
  if (c0 < inner) {
    const T* xc = x + o * N * inner + c0;
    for (int64_t n = n0 + ty; n < n1; n += TY * U) {
      // All U loads, then their uses: rows past the end repeat the last one
      // (a load under a branch of its own would be waited for there) and
      // read as -inf.
      Pack<T> p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const T* at = xc + min(n + u * TY, n1 - 1) * inner;
        if constexpr (V > 1) p[u] = load_pack_nt(at);
        else p[u].v[0] = *at;
      }
      float vals[V][U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int e = 0; e < V; ++e)
          vals[e][u] = n + u * TY < n1 ? Elem<T>::to_f32(p[u].v[e]) : -INFINITY;
      }
#pragma unroll
      for (int e = 0; e < V; ++e) {
        if constexpr (OP == 0) {
          lse_fold<U>(st[e], vals[e]);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (n + u * TY < n1) arg_step<OP == 2>(st[e], vals[e][u], (int)(n + u * TY));
        }
      }
    }
  }
  auto put = [&](int64_t col, S v) {
    const int64_t i = o * inner + col;
    if (nsplit > 1) static_cast<S*>(out)[i * nsplit + split] = v;
    else row_store<T, OP>(out, i, v);
  };
  if constexpr (TY == 1) {
    if (c0 < inner) {
#pragma unroll
      for (int e = 0; e < V; ++e) put(c0 + e, st[e]);
    }
  } else {
    __shared__ S part[TY][TX * V];
#pragma unroll
    for (int e = 0; e < V; ++e) part[ty][tx * V + e] = st[e];
    __syncthreads();
    for (int c = threadIdx.x; c < TX * V; c += 256) {
      const int64_t col = tile * TX * V + c;
      if (col >= inner) break;
      S v = part[0][c];
#pragma unroll 4
      for (int y = 1; y < TY; ++y) v = row_merge<OP>(v, part[y][c]);
      put(col, v);
    }
  }
}

// Threads across the columns: 256 where that alone fills the chip, and for a
// few rows from half a workgroup per CU on (LogSumExp bf16 [4, 128, 4096] over
// dimension 0: 5.3 us with 256, 6.7 with 64 and their merge; bf16 [8, 2^20] 8.9
// and 12.4, fp32 [2, 2^19] 4.7 and 6.8) except where a thread would store eight
// scattered indices (Argmax fp16 of that shape: 7.8 and 6.6; bf16 [8, 2^20] 13.4
// and 10.8); else 64, else 16.  With less than a workgroup per CU and six steps
// of ~2 us or more the rows are split, one step each up to two workgroups per
// CU (Argmax bf16 [3, 1000, 64]: 32 us whole, 9.7 split; 300 rows: 9.4 either
// way, and whole is one launch).  Rows past the end of a thread's last step
// repeat the last one, so that its loads are all in flight (Argmax bf16 [46,
// 276, 2113]: 38.5 us with a branch per load, 28.6 so).
struct ColPlan {
  int v, tx, nsplit;
  int64_t ntile;
};
static ColPlan plan_cols(int64_t outer, int64_t N, int64_t inner, int vec, bool arg) {
  ColPlan p{inner % vec == 0 ? vec : 1, 16, 1, 0};
  const int64_t packs = inner / p.v;
  auto blocks = [&](int tx) { return outer * ((packs + tx - 1) / tx); };
  if (packs > 64 && blocks(256) >= (N <= 8 && !(arg && p.v == 8) ? 128 : 1024)) p.tx = 256;
  else if (packs > 16 && (N <= 32 || blocks(64) >= 512)) p.tx = 64;
  p.ntile = (packs + p.tx - 1) / p.tx;
  const int64_t wg = blocks(p.tx), steps = N / (256 / p.tx * 4);
  if (wg < 256 && steps >= 6) p.nsplit = (int)std::min<int64_t>(steps, 512 / wg);
  return p;
}

template <typename T, int OP, int V>
static int launch_cols(const T* x, void* out, int64_t outer, int64_t N, int64_t inner,
                       const ColPlan& p, hipStream_t s) {
  auto go = [&](auto kernel) {
    return launch_slices(p.ntile * p.nsplit * outer, 256, [&](int64_t block0, dim3 grid) {
      kernel<<<grid, dim3(256), 0, s>>>(x, out, N, inner, p.ntile, p.nsplit, block0);
    });
  };
  if (p.tx == 256) return go(col_reduce_kernel<T, OP, V, 256>);
  if (p.tx == 64) return go(col_reduce_kernel<T, OP, V, 64>);
  return go(col_reduce_kernel<T, OP, V, 16>);
}

template <typename T, int OP>
static int launch_col_reduce(const void* xv, void* out, int64_t outer, int64_t N, int64_t inner,
                             void* ws, hipStream_t s) {
  const T* x = static_cast<const T*>(xv);
  ColPlan p = plan_cols(outer, N, inner, Elem<T>::kVec, OP != 0);
  if (p.v > 1 && !host_aligned16(x)) {  // one column per thread
    p.v = 1;
    p.ntile = (inner + p.tx - 1) / p.tx;
  }
  void* dst = p.nsplit > 1 ? ws : out;
  const int e = p.v > 1 ? launch_cols<T, OP, Elem<T>::kVec>(x, dst, outer, N, inner, p, s)
                        : launch_cols<T, OP, 1>(x, dst, outer, N, inner, p, s);
  if (e || p.nsplit == 1) return e;
  return launch_merge<T, OP>(ws, out, outer * inner, p.nsplit, s);
}

// One call: x[outer, n, inner].  kRows: rows of `inner` (outer 1); kAxis: over
// n; kEnds: over outer and inner.
enum Form { kRows, kAxis, kEnds };
struct Call {
  Form form;
  const void* x;
  void* y;
  int64_t outer, n, inner;
  void* ws;
  size_t ws_bytes;
  hipStream_t s;
};

template <typename T, int OP>
static int launch_call(const Call& c) {
  if (c.form == kAxis)
    return launch_col_reduce<T, OP>(c.x, c.y, c.outer, c.n, c.inner, c.ws, c.s);
  return launch_row_reduce<T, OP>(c.x, c.y, c.outer * c.n, c.inner, c.form == kEnds ? c.n : 0,
                                  c.ws, c.ws_bytes, c.s);
}

template <int OP>
static int dispatch_call(const Call& c, int dtype) {
  switch (dtype) {
    case TILEOPS_F32: return launch_call<float, OP>(c);
    case TILEOPS_F16: return launch_call<f16, OP>(c);
    case TILEOPS_BF16: return launch_call<bf16, OP>(c);
  }
  return TILEOPS_EINVAL;
}

static int run_call(int op, Call c, int dtype) {
  if (c.ws && !host_aligned16(c.ws)) return TILEOPS_EINVAL;
  if (!c.ws) c.ws_bytes = 0;
  switch (op) {
    case TILEOPS_LOGSUMEXP: return dispatch_call<0>(c, dtype);
    case TILEOPS_ARGMAX: return dispatch_call<1>(c, dtype);
    case TILEOPS_ARGMIN: return dispatch_call<2>(c, dtype);
  }
  return TILEOPS_EINVAL;
}

// Checks and dispatch shared by the row entry points.
static int reduce_rows(int op, const void* x, void* y, int64_t M, int64_t N, int dtype, void* ws,
                       size_t ws_bytes, hipStream_t s) {
  if (M < 0 || N <= 0 || N > INT32_MAX) return TILEOPS_ESHAPE;
  if (dtype < TILEOPS_F32 || dtype > TILEOPS_BF16) return TILEOPS_EINVAL;
  if (M == 0) return 0;
  if (!x || !y) return TILEOPS_ENULL;
  return run_call(op, Call{kRows, x, y, 1, M, N, ws, ws_bytes, s}, dtype);
}

static size_t rows_bytes(int64_t M, int64_t N, int vec, int64_t folds) {
  static_assert(sizeof(LseState) == 8 && sizeof(ArgState) == 8, "partials of 8 bytes");
  const int nsplit = short_rows(N, vec) ? 1 : plan_rows(M, N, vec).nsplit;
  return folds > 1 || nsplit > 1 ? (size_t)M * nsplit * 8 : 0;
}

}  // namespace tileops

using namespace tileops;

extern "C" int tileops_logsumexp_fwd(const void* x, void* y, int64_t M, int64_t N, int dtype,
                                     void* stream) {
  return reduce_rows(TILEOPS_LOGSUMEXP, x, y, M, N, dtype, nullptr, 0,
                     static_cast<hipStream_t>(stream));
}

extern "C" int tileops_argreduce_fwd(const void* x, int64_t* y, int64_t M, int64_t N, int dtype,
                                     int is_min, void* stream) {
  return reduce_rows(is_min ? TILEOPS_ARGMIN : TILEOPS_ARGMAX, x, y, M, N, dtype, nullptr, 0,
                     static_cast<hipStream_t>(stream));
}

extern "C" size_t tileops_reduce_workspace_bytes(int64_t M, int64_t N, int dtype) {
  if (M <= 0 || N <= 0 || N > INT32_MAX || dtype < TILEOPS_F32 || dtype > TILEOPS_BF16) return 0;
  return rows_bytes(M, N, dtype == TILEOPS_F32 ? 4 : 8, 1);
}

extern "C" int tileops_reduce_fwd(int op, const void* x, void* y, int64_t M, int64_t N, int dtype,
                                  void* ws, size_t ws_bytes, void* stream) {
  return reduce_rows(op, x, y, M, N, dtype, ws, ws_bytes, static_cast<hipStream_t>(stream));
}

extern "C" size_t tileops_reduce_axis_workspace_bytes(int op, int64_t outer, int64_t n,
                                                      int64_t inner, int ends, int dtype) {
  if (outer <= 0 || n <= 0 || inner <= 0 || dtype < TILEOPS_F32 || dtype > TILEOPS_BF16) return 0;
  const int vec = dtype == TILEOPS_F32 ? 4 : 8;
  if (ends) return rows_bytes(outer * n, inner, vec, outer);
  const int64_t nsplit = plan_cols(outer, n, inner, vec, op != TILEOPS_LOGSUMEXP).nsplit;
  return nsplit > 1 ? (size_t)(outer * inner * nsplit) * 8 : 0;
}

extern "C" int tileops_reduce_axis_fwd(int op, const void* x, void* y, int64_t outer, int64_t n,
                                       int64_t inner, int ends, int dtype, void* ws,
                                       size_t ws_bytes, void* stream) {
  if (outer < 0 || n < 0 || inner < 0) return TILEOPS_ESHAPE;
  if (n > INT32_MAX || inner > INT32_MAX || outer > INT32_MAX) return TILEOPS_ESHAPE;
  if (dtype < TILEOPS_F32 || dtype > TILEOPS_BF16) return TILEOPS_EINVAL;
  if (ends && op != TILEOPS_LOGSUMEXP) return TILEOPS_EINVAL;  // an index has no order there
  if (outer == 0 || n == 0 || inner == 0) return TILEOPS_ESHAPE;
  if (outer > INT64_MAX / n / inner) return TILEOPS_ESHAPE;
  if (!x || !y) return TILEOPS_ENULL;
  if (ws_bytes < tileops_reduce_axis_workspace_bytes(op, outer, n, inner, ends, dtype) ||
      (!ws && ws_bytes > 0))
    return TILEOPS_EWORKSPACE;
  return run_call(op, Call{ends ? kEnds : kAxis, x, y, outer, n, inner, ws, ws_bytes,
                           static_cast<hipStream_t>(stream)}, dtype);
}
