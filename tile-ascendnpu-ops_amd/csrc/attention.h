// Pieces shared by the attention kernels: MFMA operand types, the LDS swizzles
// of K and V tiles, direct-to-LDS loads and lane exchanges.
#pragma once

#include <float.h>

#include "common.h"

namespace tileops {
namespace mha {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename T> struct Mfma;
template <> struct Mfma<bf16> {
  typedef bf16x8 V8;
  __device__ __forceinline__ static f32x16 run(V8 a, V8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma<f16> {
  typedef f16x8 V8;
  __device__ __forceinline__ static f32x16 run(V8 a, V8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// K and V tiles live in LDS unpadded, rows of D / 8 16-byte chunks, chunks
// XOR-swizzled by row: K so that an MFMA operand read (16 consecutive key
// rows, one chunk each) hits 16 distinct 16-byte bank groups, V so that the
// transpose reads of a half-wavefront (4 consecutive key rows x 64 bytes)
// cover all 64 banks once.
template <int D> struct Swz {
  static constexpr int CPR = D / 8;  // chunks per row
  __host__ __device__ static constexpr int k_key(int r) { return CPR >= 16 ? (r & 15) : ((r >> 1) & 7); }
  __host__ __device__ static constexpr int v_key(int r) { return CPR == 16 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); }
};

// One 16-byte direct-to-LDS load per lane: lane l reads 16 bytes at
// `base + off` (base uniform, in SGPRs; off a per-lane byte offset) and they
// land at LDS byte address lds + 16 l.  Issued as inline assembly so that the
// compiler does not track the LDS write: every wait for these loads is
// explicit (vmcnt) and followed by a workgroup barrier before another wavefront
// reads the data.  The compiler's hazard checks do not look into inline
// assembly: the load starts with the one wait state the ISA requires after
// the SALU write of M0 that precedes it (its base comes from SALU
// arithmetic, so no VALU-to-SGPR wait is involved).
__device__ __forceinline__ void lds_dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(lds)
               : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(lds_void_ptr)p;
}

// Combine a value with the one held by the partner lane l ^ 32 (VALU lane
// swap between the two wavefront halves, no LDS round trip): the two
// outputs of v_permlane32_swap on (x, x) are x's low and high halves.
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x),
                                                  __builtin_bit_cast(unsigned, x), false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x),
                                                  __builtin_bit_cast(unsigned, x), false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}

// tanh(y) = 1 - 2 / (1 + e^{2y}), saturating to +-1 through the
// exponential's overflow / underflow (no branch)
__device__ __forceinline__ float tanh_sat(float y) {
  const float e = __builtin_amdgcn_exp2f(y * (2.0f * 1.4426950408889634f));
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + e);
}

// One attention call.
struct Problem {
  const void *q, *k, *v;
  void* o;
  float* lse;
  int B, Sq, Skv, H, Hkv, D;
  bool causal;
  float scale, softcap;
  int dtype;
};

// The key-split kernel (attention_split.hip): its best layout for these sizes
// (or the one with `nsplit` splits), whether it takes them, whether that layout
// beats mha_fwd_kernel, the scratch it uses, and the launch.
constexpr int kMaxSplit = 64;
struct SplitPlan {
  int ntile, nsplit;
  double us;
};
SplitPlan split_plan(const Problem& p, int nsplit = 0);
bool split_fits(const Problem& p, const SplitPlan& plan);
bool split_wins(const Problem& p, const SplitPlan& plan);
size_t split_bytes(const Problem& p, const SplitPlan& plan);
int split_launch(const Problem& p, const SplitPlan& plan, void* ws, hipStream_t s);

}  // namespace mha
}  // namespace tileops
