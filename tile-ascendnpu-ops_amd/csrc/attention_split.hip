// Attention forward for few query rows against many keys (a decode step, a
// short chunk appended to a cache), BSHD layout: the keys are split.
//
// mha_fwd_kernel takes 256 query rows of one head per workgroup, so a decode
// step fills one row in 256 and reads a grouped head's K and V once per query
// head.  Here a tile is 32 query rows of one K / V head -- the queries of all
// heads of its group, token major -- and a workgroup walks one split of the
// keys: every wavefront streams its own 32-key blocks of K and V through a
// private pair of LDS slots by direct-to-LDS loads (whole rows, no workgroup
// barrier in the loop; while block i is computed, V of block i, block i + 1
// and K of block i + 2 are in flight: 96 KB per CU at D = 128), with the
// products, swizzles and transpose reads of mha_fwd_kernel.  The wavefronts of
// a workgroup meet in LDS, and the splits in mha_combine_kernel, through fp32
// partial outputs and (max, sum) per row.  A decode step is bound by reading K
// and V once: B8 H32/8 S1 x 8191 D128 bf16 took 176 us with mha_fwd_kernel and
// takes 50.5 (5.3 TB/s) here; B1 S1 x 32768 555 -> 33.5, B1 S128 x 8192 139 ->
// 56, B1 H8 S256 x 256 13.6 -> 10.2.
#include <algorithm>

#include "attention.h"

namespace tileops {
namespace mha {

template <int D> struct SplitShape {
  static constexpr int DP = D <= 64 ? 64 : D <= 128 ? 128 : 256;  // LDS row width
  static constexpr int NW = DP == 256 ? 2 : 4;                    // wavefronts
  static constexpr int TILE = 32 * DP;                            // elements of a K or V block
  static constexpr int WIN = TILE / 512;                          // 1 KB windows per block
  static constexpr int WGS = DP == 64 ? 2 : 1;                    // workgroups per CU (LDS)
};

// s_waitcnt vmcnt(N), in program order with the LDS reads around it.
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt is six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// As lds_dma16, with the wait states that a VALU write of an SGPR read by a
// vector memory instruction needs (the base may come from v_readfirstlane).
// NT: keys and values that one workgroup alone reads do not stay in L2
// (attention_decode's shape above: 59.4 us with plain loads, 51.4 so).
template <bool NT>
__device__ __forceinline__ void lds_dma16_any(const void* base, uint32_t off, uint32_t lds) {
  if constexpr (NT)
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(off), "s"(base), "{m0}"(lds)
                 : "memory");
  else
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(lds)
                 : "memory");
}

struct SplitArgs {
  const void *q, *k, *v;
  void* o;
  float* lse;
  float* part;  // [nsplit][rows][D] partial outputs, then [nsplit][rows][2] (max, sum)
  int B, Sq, Skv, H, Hkv;
  int causal;
  float scale_log2, cap_scale, cap_log2;  // cap_log2 > 0: soft-capped scores
  int ntile, nsplit;                      // row tiles per K / V head, key splits
};

template <typename T, int D, bool NT>
__global__ __launch_bounds__(64 * SplitShape<D>::NW) void mha_split_kernel(SplitArgs A) {
  typedef typename Mfma<T>::V8 V8;
  typedef SplitShape<D> Sh;
  constexpr int DP = Sh::DP, NW = Sh::NW, TILE = Sh::TILE, WIN = Sh::WIN;
  constexpr int KSTEPS = D / 16, DBLK = D / 32, CPR = DP / 8, RCPR = D / 8;
  __shared__ __attribute__((aligned(1024))) T lds[NW * 4 * TILE];  // per wave: K0 K1 V0 V1
  __shared__ float stat[NW][2][32];

  const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // workgroup i runs on XCD i % 8: the row tiles of one (head, split) are
  // neighbours on one XCD, so that its K and V are read from HBM once
  int id = blockIdx.x;
  const int nblk = (int)gridDim.x;
  if ((nblk & 7) == 0) id = (id & 7) * (nblk >> 3) + (id >> 3);
  const int tile = id % A.ntile;
  id /= A.ntile;
  const int split = id % A.nsplit;
  id /= A.nsplit;
  const int hk = id % A.Hkv, b = id / A.Hkv;
  const int G = A.H / A.Hkv, R = A.Sq * G, off = A.Skv - A.Sq;

  // this lane's query row: token sq, head hk G + g
  const int r = tile * 32 + col;
  const int rc = min(r, R - 1), sq = rc / G;
  const int64_t qrow = ((int64_t)b * A.Sq + sq) * A.H + hk * G + (rc - sq * G);
  const T* qp = static_cast<const T*>(A.q) + qrow * D + half * 8;
  V8 qreg[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    const u32x4 raw = *reinterpret_cast<const u32x4*>(qp + ks * 16);
    qreg[ks] = *reinterpret_cast<const V8*>(&raw);
  }
  // last visible key of this lane's row, of the tile's first row and of its last
  const int lim = A.causal ? min(A.Skv - 1, sq + off) : A.Skv - 1;
  const int lim_lo = A.causal ? (tile * 32) / G + off : A.Skv - 1;
  const int kv_end = A.causal ? min(A.Skv, (min(tile * 32 + 31, R - 1)) / G + off + 1) : A.Skv;
  // this split's 32-key blocks, dealt to the wavefronts in turn
  const int nb_all = (kv_end + 31) / 32, bps = (nb_all + A.nsplit - 1) / A.nsplit;
  const int blk0 = split * bps + wave, blk_end = min(nb_all, (split + 1) * bps);
  const int n = blk0 < blk_end ? (blk_end - blk0 + NW - 1) / NW : 0;

  // Window i of a block: lane l fills chunk 64 i + l of the swizzled image
  // (row = chunk / CPR); rows past the last key repeat it (masked below), and
  // the padding chunks of D = 96 and 192 a real chunk (never read).
  const int64_t kv_row = (int64_t)A.Hkv * D;
  const T* kbase = static_cast<const T*>(A.k) + (int64_t)b * A.Skv * kv_row + (int64_t)hk * D;
  const T* vbase = static_cast<const T*>(A.v) + (int64_t)b * A.Skv * kv_row + (int64_t)hk * D;
  const uint32_t row_bytes = (uint32_t)(kv_row * sizeof(T));
  T* const mine = lds + wave * 4 * TILE;
  auto load = [&](const T* src0, T* dst, int i, bool is_v) __attribute__((always_inline)) {
    const int key0 = (blk0 + i * NW) * 32;
    const T* src = src0 + (int64_t)key0 * kv_row;
    const int rmax = min(31, A.Skv - 1 - key0);
    const uint32_t base = lds_addr(dst);
#pragma unroll
    for (int w = 0; w < WIN; ++w) {
      const int ch = w * 64 + lane, row = ch / CPR, p = ch % CPR;
      const int c = p ^ (is_v ? Swz<DP>::v_key(row) : Swz<DP>::k_key(row));
      const int gc = c < RCPR ? c : c - (CPR - RCPR);
      lds_dma16_any<NT>(src, (uint32_t)min(row, rmax) * row_bytes + (uint32_t)(gc * 16), base + w * 1024);
    }
  };
  auto load_k = [&](int i) __attribute__((always_inline)) { load(kbase, mine + (i & 1) * TILE, i, false); };
  auto load_v = [&](int i) __attribute__((always_inline)) { load(vbase, mine + (2 + (i & 1)) * TILE, i, true); };

  // operand read addresses (as in mha_fwd_kernel)
  const uint32_t kbx = lds_addr(mine) + (uint32_t)(col * DP * 2) +
                       16u * (uint32_t)(half ^ Swz<DP>::k_key(col));
  const int grp16 = lane >> 4, j16 = lane & 15;
  const int vrow = 4 * (grp16 >> 1) + (j16 >> 2), vdim = 16 * (grp16 & 1) + 4 * (j16 & 3);
  const uint32_t vbx =
      lds_addr(mine) + 2 * TILE * 2 +
      (uint32_t)((vrow * DP + ((((vdim >> 3) ^ Swz<DP>::v_key(vrow)) << 3) | (vdim & 7))) * 2);
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  typedef __attribute__((address_space(3))) V8 lds_v8;

  f32x16 acc_o[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i) acc_o[i] = f32x16{};
  float m_run = -INFINITY, l_run = 0.0f;  // m in raw scores (capped: log2 units)

  if (n > 0) load_k(0), load_v(0);
  if (n > 1) load_k(1), load_v(1);
  for (int i = 0; i < n; ++i) {
    // K(i) has landed: V(i), K(i + 1), V(i + 1) may be in flight
    if (i + 1 < n) wait_vm<3 * WIN>();
    else wait_vm<WIN>();
    f32x16 s = {};
    {
      const uint32_t kb = kbx + (uint32_t)((i & 1) * TILE * 2);
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
        s = Mfma<T>::run(*(lds_v8*)(uintptr_t)(kb ^ (32u * (uint32_t)ks)), qreg[ks], s);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // K(i) is read
    if (i + 2 < n) load_k(i + 2);

    if (A.cap_log2 > 0.0f) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = A.cap_log2 * tanh_sat(s[e] * A.cap_scale);
    }
    const int kv0 = (blk0 + i * NW) * 32;
    if (kv0 + 31 > lim_lo || kv0 + 31 >= A.Skv) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int kv = kv0 + (e >> 2) * 8 + (e & 3) + 4 * half;
        s[e] = kv > lim ? -INFINITY : s[e];
      }
    }
    float tm[4] = {s[0], s[1], s[2], s[3]};
#pragma unroll
    for (int e = 4; e < 16; ++e) tm[e & 3] = fmaxf(tm[e & 3], s[e]);
    const float m_new = fmaxf(m_run, pair_max(fmaxf(fmaxf(tm[0], tm[1]), fmaxf(tm[2], tm[3]))));
    if (__any(m_new > m_run)) {
      const float alpha =
          m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_new) * A.scale_log2);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DBLK; ++db) {
#pragma unroll
        for (int e = 0; e < 16; ++e) acc_o[db][e] *= alpha;
      }
      m_run = m_new;
    }
    const float neg = m_run == -INFINITY ? 0.0f : -m_run * A.scale_log2;
    V8 pb[2];
    float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float p = __builtin_amdgcn_exp2f(fmaf(s[e], A.scale_log2, neg));
      ps[e & 3] += p;
      pb[e >> 3][e & 7] = (T)p;
    }
    l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);

    // V(i) has landed
    if (i + 2 < n) wait_vm<3 * WIN>();
    else if (i + 1 < n) wait_vm<2 * WIN>();
    else wait_vm<0>();
    {
      const uint32_t vb0 = vbx + (uint32_t)((i & 1) * TILE * 2);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int db = 0; db < DBLK; ++db) {
          const uint32_t vb = (vb0 ^ (64u * (uint32_t)db)) + (uint32_t)(16 * ks * DP * 2);
          const v4i16 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(uintptr_t)vb);
          const v4i16 x1 =
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(uintptr_t)(vb + 8 * DP * 2));
          const u32x2 y0 = __builtin_bit_cast(u32x2, x0), y1 = __builtin_bit_cast(u32x2, x1);
          const u32x4 w = {y0.x, y0.y, y1.x, y1.y};
          acc_o[db] = Mfma<T>::run(__builtin_bit_cast(V8, w), pb[ks], acc_o[db]);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // V(i) is read
    if (i + 2 < n) load_v(i + 2);
  }

  // --- the wavefronts' partials meet in LDS: statistics first, then the
  // outputs on the common max, [wave][dim][row] with rows padded to 33 (each wavefront's loads have
  // landed and its tiles are free)
  const float l_row = pair_sum(l_run);
  if (half == 0) {
    stat[wave][0][col] = m_run;
    stat[wave][1][col] = l_row;
  }
  __syncthreads();
  float m = stat[0][0][col];
#pragma unroll
  for (int w = 1; w < NW; ++w) m = fmaxf(m, stat[w][0][col]);
  auto factor = [&](float mw) {
    return mw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mw - m) * A.scale_log2);
  };
  float l = 0.0f;
#pragma unroll
  for (int w = 0; w < NW; ++w) l += stat[w][1][col] * factor(stat[w][0][col]);
  static_assert(4 * TILE * 2 >= 33 * D * 4, "partial outputs fit a wavefront's tiles");
  float* const ob = reinterpret_cast<float*>(lds);
  constexpr int OBW = 4 * TILE / 2;  // floats per wavefront region
  {
    const float f = factor(m_run);
#pragma unroll
    for (int db = 0; db < DBLK; ++db) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        ob[wave * OBW + (db * 32 + (e >> 2) * 8 + half * 4 + (e & 3)) * 33 + col] =
            acc_o[db][e] * f;
    }
  }
  // row statistics of the workgroup, and the factor of its outputs
  const bool last = A.nsplit == 1;
  const float inv_l = l > 0.0f ? 1.0f / l : 0.0f;
  const int64_t rows = (int64_t)A.B * A.Sq * A.H;
  if (wave == 0 && half == 0 && r < R) {
    if (last) {
      const int64_t bh = (int64_t)b * A.H + hk * G + (rc - sq * G);
      A.lse[bh * A.Sq + sq] = l > 0.0f ? m * A.scale_log2 + __builtin_amdgcn_logf(l) : -INFINITY;
    } else {
      float* st = A.part + (int64_t)A.nsplit * rows * D + ((int64_t)split * rows + qrow) * 2;
      st[0] = m * A.scale_log2;
      st[1] = l;
    }
  }
  __syncthreads();  // outputs written; stat is read no more below
  if (wave == 0 && half == 0) stat[0][1][col] = inv_l;
  __syncthreads();
  // sum over the wavefronts, row by row: lanes run over dims
  for (int rr = wave; rr < 32; rr += NW) {
    const int row = tile * 32 + rr;
    if (row >= R) break;
    const int s_ = row / G;
    const int64_t grow = ((int64_t)b * A.Sq + s_) * A.H + hk * G + (row - s_ * G);
    for (int d = lane; d < D; d += 64) {
      float v = ob[d * 33 + rr];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += ob[w * OBW + d * 33 + rr];
      if (last) static_cast<T*>(A.o)[grow * D + d] = (T)(v * stat[0][1][rr]);
      else A.part[((int64_t)split * rows + grow) * D + d] = v;
    }
  }
}

// The splits' partial outputs of each query row (one wavefront per row).
template <typename T, int D>
__global__ __launch_bounds__(256) void mha_combine_kernel(SplitArgs A) {
  const int lane = threadIdx.x & 63;
  const int64_t rows = (int64_t)A.B * A.Sq * A.H;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* st = A.part + (int64_t)A.nsplit * rows * D;
  float mi = -INFINITY, li = 0.0f;  // split `lane` (nsplit <= 64)
  if (lane < A.nsplit) {
    mi = st[((int64_t)lane * rows + row) * 2];
    li = st[((int64_t)lane * rows + row) * 2 + 1];
  }
  const float m = wave_max(mi);
  const float w = mi == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mi - m);
  const float l = wave_sum(li * w);
  constexpr int E = (D + 63) / 64;
  float acc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = 0.0f;
  for (int i = 0; i < A.nsplit; ++i) {
    const float wi = __shfl(w, i, 64);
    const float* po = A.part + ((int64_t)i * rows + row) * D;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (e * 64 + lane < D) acc[e] = fmaf(wi, po[e * 64 + lane], acc[e]);
  }
  const float inv_l = l > 0.0f ? 1.0f / l : 0.0f;
  T* o = static_cast<T*>(A.o) + row * D;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (e * 64 + lane < D) o[e * 64 + lane] = (T)(acc[e] * inv_l);
  if (lane == 0) {
    const int64_t h = row % A.H, bs = row / A.H, sq = bs % A.Sq, b = bs / A.Sq;
    A.lse[(b * A.H + h) * A.Sq + sq] = l > 0.0f ? m + __builtin_amdgcn_logf(l) : -INFINITY;
  }
}

// ---------------------------------------------------------------------------
// When and how far to split, from estimated times in us.  The rates are fitted
// to 1350 random shapes timed with mha_fwd_kernel and with up to twelve split
// counts (every head dimension, 1 to 1024 queries, 16 to 32768 keys, 1 to 64
// heads; the estimates are off by 11 and 8 %).  The split kernel is taken where
// it is expected to be at least a tenth faster, a fifth at head dimensions 192
// and 256.  One of those shapes is then slower than with mha_fwd_kernel (6 %);
// over all, calls are 1.58 times faster (geometric mean), and would be 1.60
// with the faster kernel every time.  On 700 others: one slower (15 %), 1.60
// times.  (Rates from 36 shapes of head dimensions 64 and 128, one fixed cost
// for all, made 100 of 900 shapes slower: B34 S94 H64/8 D192 took 375 us where
// mha_fwd_kernel takes 134, B64 S64 H32 D128 115 where it takes 77.)
// ---------------------------------------------------------------------------
struct Rates {
  int D;
  double main_fixed, main_tile;             // mha_fwd_kernel: a workgroup, and a key tile of it
  double split_fixed, split_rows, split_step;  // a workgroup, its 32 rows' outputs, a step
};
static const Rates& rates_of(int D) {
  static const Rates rates[] = {{64, 5.1, 0.93, 0.9, 1.9, 1.15},
                                {96, 7.2, 1.97, 1.7, 3.1, 1.4},
                                {128, 7.5, 2.22, 2.2, 3.0, 1.45},
                                {192, 5.9, 1.43, 2.4, 6.6, 1.95},
                                {256, 6.0, 1.83, 3.4, 6.5, 2.35}};
  for (const Rates& r : rates)
    if (r.D >= D) return r;
  return rates[4];
}

// What an eager call of `us` on the GPU costs: it is no shorter than its host
// path, ~10.4 us with one launch and ~14.5 with two and scratch.  Equal costs
// go by the GPU time.
static double call_cost(double us, bool two_launches) {
  return std::max(us, two_launches ? 14.5 : 10.4) + 1e-3 * us;
}

// mha_fwd_kernel: a workgroup per CU and round; the longest block where every
// block is resident at once, else the mean one.  Its loads of a decode step's
// keys are HBM traffic it does not hide (3.9 TB/s).
static double main_us(const Problem& p) {
  const Rates& r = rates_of(p.D);
  const int64_t cus = device_cu_count();
  const int64_t blocks = ((int64_t)p.Sq + 255) / 256 * p.H * p.B * (p.D >= 192 ? 2 : 1);
  const double whole = (double)((blocks + cus - 1) / cus);
  const double rounds = blocks <= 3 * cus ? whole : std::min(whole, (double)blocks / cus + 0.5);
  const int keys = p.causal && rounds > 1.0 ? p.Skv - std::max(p.Sq - 256, 0) / 2 : p.Skv;
  const int bn = p.D == 96 || p.D == 128 ? 128 : 64;
  const double hbm = (double)p.B * p.Hkv * p.Skv * p.D * 4.0 / 3.9e6;
  return 0.8 + r.main_fixed * rounds + std::max(rounds * r.main_tile * ((keys + bn - 1) / bn), hbm);
}

// mha_split_kernel: a step is one 32-key block per wavefront, bound by its own
// chain of loads and products or its share of HBM (7.9 TB/s of blocks, each
// read once for all row tiles; where two workgroups share some CUs those set the
// time, as if all did); then the combination, with its launch, a few loads per
// split and row, and the partial outputs' bytes.
SplitPlan split_plan(const Problem& p, int nsplit) {
  const int64_t R = (int64_t)p.Sq * (p.H / p.Hkv);
  SplitPlan best{(int)((R + 31) / 32), 1, 1e30};
  if (nsplit > 0) {
    best.nsplit = nsplit;
    return best;
  }
  const Rates& r = rates_of(p.D);
  const int64_t base = (int64_t)p.B * p.Hkv * best.ntile;
  const int nb = (p.Skv + 31) / 32;
  const int nw = p.D > 128 ? 2 : 4, wgs = p.D <= 64 ? 2 : 1;
  const int64_t cus = device_cu_count(), slots = cus * wgs;
  const double bytes = 32.0 * (p.D <= 64 ? 64 : p.D <= 128 ? 128 : 256) * 4 * nw;
  const double hbm = bytes / 7.9e6 / best.ntile;
  const double fixed = r.split_fixed + r.split_rows * std::min<int64_t>(R, 32) / 32.0;
  const double part = 0.25 + (double)p.B * p.Sq * p.H * p.D * 4.0 / 3.7e6;
  double least = 0.0;  // call_cost of `best`
  for (int ns = 1; ns <= kMaxSplit && ns <= (nb + nw - 1) / nw; ++ns) {
    const int64_t wg = base * ns, rounds = (wg + slots - 1) / slots;
    const int steps = ((nb + ns - 1) / ns + nw - 1) / nw;
    const double step = std::max(r.split_step, hbm * (wg <= cus ? wg : slots));
    const double us = 2.6 + rounds * (fixed + steps * step) + (ns > 1 ? 3.2 + part * ns : 0.0);
    const double cost = call_cost(us, ns > 1);
    if (ns == 1 || cost < least) best.nsplit = ns, best.us = us, least = cost;
  }
  return best;
}

size_t split_bytes(const Problem& p, const SplitPlan& s) {
  if (s.nsplit == 1) return 0;
  return (size_t)s.nsplit * p.B * p.Sq * p.H * (size_t)(p.D + 2) * sizeof(float);
}

bool split_fits(const Problem& p, const SplitPlan& s) {
  if (!(p.scale > 0.0f)) return false;  // the running max is of raw scores
  // at most 2^32 - 1 threads a launch: this kernel's and the combining one's
  // (mha_fwd_kernel takes eight row tiles in 512 threads)
  const int64_t wgs = (int64_t)p.B * p.Hkv * s.ntile * s.nsplit, rows = (int64_t)p.B * p.Sq * p.H;
  if (wgs * (p.D > 128 ? 128 : 256) > (int64_t)UINT32_MAX) return false;
  if (s.nsplit > 1 && (rows + 3) / 4 * 256 > (int64_t)UINT32_MAX) return false;
  if ((int64_t)p.Sq * (p.H / p.Hkv) > (int64_t)INT32_MAX) return false;
  if ((int64_t)p.Hkv * p.D * 2 * 32 > (int64_t)UINT32_MAX) return false;
  return true;
}

bool split_wins(const Problem& p, const SplitPlan& s) {
  const double main = main_us(p);
  return split_fits(p, s) && s.us < (p.D > 128 ? 0.8 : 0.9) * main &&
         call_cost(s.us, s.nsplit > 1) < call_cost(main, false);
}

template <typename T, int D>
static int launch(const SplitArgs& a, const SplitPlan& s, hipStream_t st) {
  const unsigned grid = (unsigned)((int64_t)a.B * a.Hkv * s.ntile * s.nsplit);
  const dim3 block(64 * SplitShape<D>::NW);
  if (a.ntile == 1) mha_split_kernel<T, D, true><<<dim3(grid), block, 0, st>>>(a);
  else mha_split_kernel<T, D, false><<<dim3(grid), block, 0, st>>>(a);
  if (s.nsplit > 1) {
    if (int e = launch_status()) return e;
    const int64_t rows = (int64_t)a.B * a.Sq * a.H;
    mha_combine_kernel<T, D><<<dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st>>>(a);
  }
  return launch_status();
}

template <typename T>
static int launch_d(int D, const SplitArgs& a, const SplitPlan& s, hipStream_t st) {
  switch (D) {
    case 64: return launch<T, 64>(a, s, st);
    case 96: return launch<T, 96>(a, s, st);
    case 128: return launch<T, 128>(a, s, st);
    case 192: return launch<T, 192>(a, s, st);
    case 256: return launch<T, 256>(a, s, st);
  }
  return TILEOPS_ESHAPE;
}

int split_launch(const Problem& p, const SplitPlan& s, void* ws, hipStream_t st) {
  constexpr float kLog2e = 1.4426950408889634f;
  SplitArgs a{p.q, p.k, p.v, p.o, p.lse, static_cast<float*>(ws), p.B, p.Sq, p.Skv, p.H, p.Hkv,
              p.causal ? 1 : 0, p.scale * kLog2e, 0.0f, 0.0f, s.ntile, s.nsplit};
  if (p.softcap > 0.0f) {  // scores in log2 units from the cap on
    a.scale_log2 = 1.0f;
    a.cap_scale = p.scale / p.softcap;
    a.cap_log2 = p.softcap * kLog2e;
  }
  return p.dtype == TILEOPS_BF16 ? launch_d<bf16>(p.D, a, s, st) : launch_d<f16>(p.D, a, s, st);
}

}  // namespace mha
}  // namespace tileops
