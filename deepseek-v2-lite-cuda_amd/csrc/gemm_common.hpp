// Device helpers shared by the grouped GEMM kernels (gemm.hip, gemm_mid.hip).
#pragma once

#include "dsk_common.hpp"

namespace dsk {

constexpr int kMaxGroups = 128;
constexpr int kLdsPerCU = 160 * 1024;

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void global_void_t;

// silu(x) = x / (1 + e^-x) with the hardware reciprocal (1 ulp), ample for a
// result that is rounded to bf16.
__device__ __forceinline__ float silu_f(float x) {
  return x * __builtin_amdgcn_rcpf(1.f + __expf(-x));
}

// Reads an accumulator register where it is used: the epilogue then moves
// the accumulators to VGPRs a few at a time instead of all at once.
__device__ __forceinline__ float acc_read(float a) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}

// 16-byte slot of (row, logical chunk) in a tile of CPR-chunk LDS rows.
template <int CPR>
__device__ __forceinline__ int lds_swz(int row, int chunk) {
  if constexpr (CPR == 8) return row * 8 + (chunk ^ (row & 7) ^ ((row >> 3) & 1));
  else return row * 4 + (chunk ^ ((row >> 2) & 3));
}

}  // namespace dsk
