// The merge of the partial results that decode attention leaves when a request's keys are cut into
// runs: out = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M) with M = max_s m_s, for four
// consecutive dims of one (request, head). Used by the kernels that merge on their own way (the
// o projection of very few rows, the last workgroup of a decode attention launch); sums in the
// order of attention_merge_kernel, so that all three give the same bits: the denominators pairwise
// as its butterfly adds them (lanes 8 apart, then 4, 2, 1), the outputs run by run.
#pragma once
#include "common.h"

#define MERGE_SPLITS 16  // the most runs of keys that merged_quad takes

typedef float merge_float2 __attribute__((ext_vector_type(2)));
typedef float merge_float4 __attribute__((ext_vector_type(4)));

// What one workgroup of a launch hands to another goes through memory at the device's scope, past
// the caches that are private to a part of the chip: buffer loads and stores with the sc1 bit
// (bit 4 of the builtins' cache policy on gfx940 and later), 8 or 16 bytes a lane. The resource
// spans the whole address range behind the pointer (offsets are 32-bit byte offsets).
typedef unsigned merge_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned merge_u32x2 __attribute__((ext_vector_type(2)));
constexpr int DEVICE_SCOPE = 1 << 4;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t device_scope_buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffffu, 0x00020000);
}
__device__ __forceinline__ merge_float4 device_load4(__amdgpu_buffer_rsrc_t r, unsigned byte_offset) {
  union {
    merge_u32x4 raw;
    merge_float4 f;
  } u;
  u.raw = __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_offset, 0, DEVICE_SCOPE);
  return u.f;
}
__device__ __forceinline__ merge_float2 device_load2(__amdgpu_buffer_rsrc_t r, unsigned byte_offset) {
  union {
    merge_u32x2 raw;
    merge_float2 f;
  } u;
  u.raw = __builtin_amdgcn_raw_buffer_load_b64(r, (int)byte_offset, 0, DEVICE_SCOPE);
  return u.f;
}
__device__ __forceinline__ void device_store4(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, merge_float4 v) {
  union {
    merge_u32x4 raw;
    merge_float4 f;
  } u;
  u.f = v;
  __builtin_amdgcn_raw_buffer_store_b128(u.raw, r, (int)byte_offset, 0, DEVICE_SCOPE);
}
__device__ __forceinline__ void device_store2(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, merge_float2 v) {
  union {
    merge_u32x2 raw;
    merge_float2 f;
  } u;
  u.f = v;
  __builtin_amdgcn_raw_buffer_store_b64(u.raw, r, (int)byte_offset, 0, DEVICE_SCOPE);
}

// part_o [.. slots][head_dim], part_ml [.. slots][2]; `base`: the first of the S slots of this
// (request, head); d: the first of the four dims. All loads are asked for before the first is used
// (`ask`), so that the caller may ask for other things before it has them added up (`merged`).
// SAME_LAUNCH: the partial results were stored by other workgroups of this launch (each array
// under 4 GB).
// MOST: 2, 4, 8 or 16, no fewer than the S runs. (The kernels take the least: written out for sixteen runs the sums of two are 700
// cycles of a chain that nothing hides. What is added for runs that are not there are zeros, so the bits do not depend on it.)
template <int MOST, bool SAME_LAUNCH = false>
struct MergeQuad {
  static constexpr int RUNS = MOST;
  merge_float2 ml[MOST];
  merge_float4 po[MOST];

  // (The statistics first: the weights are made from them while the sums are on their way. A run that is not there: the last again,
  // which counts as nothing.)
  __device__ __forceinline__ void ask(const float* part_o, const float* part_ml, int64_t base, int S, int head_dim, int d) {
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
      const int64_t slot = base + min(j, S - 1);
      if constexpr (SAME_LAUNCH) ml[j] = device_load2(device_scope_buffer(part_ml), (unsigned)(slot * 2 * 4));
      else ml[j] = *reinterpret_cast<const merge_float2*>(part_ml + slot * 2);
    }
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
      const int64_t slot = base + min(j, S - 1);
      if constexpr (SAME_LAUNCH) po[j] = device_load4(device_scope_buffer(part_o), (unsigned)((slot * head_dim + d) * 4));
      else po[j] = *reinterpret_cast<const merge_float4*>(part_o + slot * head_dim + d);
    }
  }

  __device__ __forceinline__ merge_float4 merged(int S) const {
    float m_all = -INFINITY;
#pragma unroll
    for (int j = 0; j < MOST; ++j) m_all = fmaxf(m_all, ml[j][0]);
    const float m_safe = m_all == -INFINITY ? 0.f : m_all;
    float wgt[MOST], t[MOST];
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
      wgt[j] = j < S ? __builtin_amdgcn_exp2f(ml[j][0] - m_safe) : 0.f;
      t[j] = j < S ? __fmul_rn(ml[j][1], wgt[j]) : 0.f;
    }
#pragma unroll
    for (int h = MOST / 2; h > 0; h >>= 1)
#pragma unroll
      for (int j = 0; j < h; ++j) t[j] = __fadd_rn(t[j], t[j + h]);
    const float inv = t[0] > 0.f ? 1.f / t[0] : 0.f;
    merge_float4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < MOST; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = j < S ? __fmaf_rn(po[j][i], wgt[j], acc[i]) : acc[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = __fmul_rn(acc[i], inv);
    return acc;
  }
};

// MOST: 8 or 16, no fewer than the S runs, and the loads of so many are on their way at once.
template <bool SAME_LAUNCH = false, int MOST = MERGE_SPLITS>
__device__ __forceinline__ merge_float4 merged_quad(const float* part_o, const float* part_ml, int64_t base, int S,
                                                    int head_dim, int d) {
  auto merge = [&](auto parts) __attribute__((always_inline)) {
    // (Left to itself the compiler may save registers and wait for a run at a time, or take what the cases below have in common, their
    // first runs, out of them and wait for that: one request of 4,000 keys in 16 runs, us, so and now, heads of 32 8.0 and 6.7, of 48 6.9
    // and 5.9, of 64 7.3 and 7.2.)
    asm volatile("; %0 runs" ::"i"(decltype(parts)::RUNS) : "memory");
    parts.ask(part_o, part_ml, base, S, head_dim, d);
    __builtin_amdgcn_sched_barrier(0);
    return parts.merged(S);
  };
  if (S <= 2) return merge(MergeQuad<2, SAME_LAUNCH>());
  if (S <= 4) return merge(MergeQuad<4, SAME_LAUNCH>());
  if (MOST == 8 || S <= 8) return merge(MergeQuad<8, SAME_LAUNCH>());
  return merge(MergeQuad<16, SAME_LAUNCH>());
}
