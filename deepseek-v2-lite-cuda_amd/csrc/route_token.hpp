// Softmax and top-K selection of one token on a 16-lane row, shared by the
// route kernel (moe_route.hip) and the first GEMM of a one-token step, which
// routes for itself (gemv.hip), so both pick the same experts with the same
// weights, bit for bit.
#pragma once

#include <math.h>

#include "dsk_common.hpp"

namespace dsk {

constexpr int kMaxGateParts = 4;  // partial gate-sum planes a logit may be split into

// Order-preserving image of a float as an unsigned key (larger float, larger key; -0 and
// +0 alike; NaN as -inf) and back. Every key is above 0, which is left for "not a choice".
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t u = __float_as_uint(v == v ? v + 0.f : -INFINITY);
  return (u >> 31) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float order_value(uint32_t key) {
  return __uint_as_float((key >> 31) ? (key & 0x7fffffffu) : ~key);
}

// Token t on one 16-lane row: lane j of the row holds the logits of experts j,
// j+16, j+32, j+48, so every reduction is a 4-value local step plus a 16-lane
// DPP step. The logits are the sum of n_parts partial planes (K slices of the
// gate GEMM) in plane order, plus the optional per-expert bias. Lane j < K of
// the row gets the j-th pick (my_e, my_w: expert and softmax probability,
// descending, NaN as -inf, ties to the lower index). active: t < T (uniform
// over the row); wave_active: some row of the wave is active (the selection
// loop has wave-wide DPP steps).
//
// A workgroup of 64 tokens keeps 4 waves on each SIMD, so its time is the count of the
// loop's instructions. The logits are compared as unsigned keys: a pick is two max3, a
// 16-lane max, the lowest index that holds it and four selects, about 30 instructions
// against more than 100 with flags and float compares beside each value, and the pick's
// probability is taken from its key once, after the loop. Route kernel at 16 tokens
// 6.1 -> 4.8 us, at 61 and 1000 (16 waves a workgroup) 9.6 and 10.0 -> 6.3 and 6.7 us.
__device__ __forceinline__ void route_token(const float* __restrict__ logits, int64_t ld,
                                            int n_parts, int64_t part_stride,
                                            const float* __restrict__ bias, int t, bool active,
                                            bool wave_active, int E, int K, int lane, int& my_e,
                                            float& my_w) {
  const int j = lane & 15;
  float xv[4];
  uint32_t key[4];  // 0: padding expert, or taken
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = j + 16 * q;
    float v = -INFINITY;
    if (active && e < E) {
      // all plane loads issued first, then summed in plane order
      const float* src = logits + (int64_t)t * ld + e;
      float pv[kMaxGateParts];
#pragma unroll
      for (int s = 0; s < kMaxGateParts; ++s) pv[s] = s < n_parts ? src[s * part_stride] : 0.f;
      v = pv[0];
#pragma unroll
      for (int s = 1; s < kMaxGateParts; ++s)
        if (s < n_parts) v += pv[s];
      if (bias != nullptr) v += bias[e];
    }
    xv[q] = v;
    key[q] = e < E ? order_key(v) : 0u;
  }
  const float mx = row16_max(fmaxf(fmaxf(xv[0], xv[1]), fmaxf(xv[2], xv[3])));
  float ex[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) ex[q] = j + 16 * q < E ? expf(xv[q] - mx) : 0.f;
  const float sum = row16_sum((ex[0] + ex[1]) + (ex[2] + ex[3]));
  my_e = -1;
  uint32_t my_key = 0;
  for (int k = 0; k < K && wave_active; ++k) {
    const uint32_t m = row16_max(max(max(key[0], key[1]), max(key[2], key[3])));
    // the lowest expert that holds it
    int at = 64;
#pragma unroll
    for (int q = 3; q >= 0; --q) at = key[q] == m ? j + 16 * q : at;
    const int win = row16_min(at);
#pragma unroll
    for (int q = 0; q < 4; ++q) key[q] = j + 16 * q == win ? 0u : key[q];
    my_e = j == k ? win : my_e;
    my_key = j == k ? m : my_key;
  }
  my_w = my_e >= 0 ? expf(order_value(my_key) - mx) / sum : 0.f;
}


// Routing of one chunk of kRouteChunk tokens by one workgroup, four tokens per
// wave (one per 16-lane row; the workgroup needs a wave per four tokens of the
// chunk). Writes topk idx / weights, the chunk histogram, and (optionally) each
// (token, k)'s rank inside its chunk. With a single chunk (T <= 64) it also
// finishes the job that the scan and permutation kernels do for larger T:
// counts, offsets (including the rows of the always-on groups appended after
// the routed ones), token_map and slot_of.
constexpr int kRouteChunk = 64;  // tokens per routing workgroup (= mask width)

__device__ __forceinline__ void route_chunk_body(
    const float* __restrict__ logits, int64_t ld, int n_parts, int64_t part_stride,
    const float* __restrict__ bias, int T, int E, int K,
    int32_t* __restrict__ topk_idx, float* __restrict__ topk_w,
    int32_t* __restrict__ blk_hist, int32_t* __restrict__ local_rank,
    int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ token_map, int32_t* __restrict__ slot_of,
    int n_extra_groups, int chunk, bool single_chunk) {
  __shared__ unsigned long long s_mask[64];
  __shared__ int s_off[64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (tid < 64) s_mask[tid] = 0ull;
  __syncthreads();

  const int t0 = chunk * kRouteChunk;
  // Four tokens per wave at once: the 16 lanes of row g hold token
  // tl = 4 * wave + g (route_token).
  const int g = lane >> 4, j = lane & 15;
  const int tl = 4 * wave + g;
  const int t = t0 + tl;
  const bool active = t < T;  // uniform over the 16-lane row
  // waves whose four rows are all past T skip the selection
  const bool wave_active = t0 + 4 * wave < T;
  int my_e;
  float my_w;
  route_token(logits, ld, n_parts, part_stride, bias, t, active, wave_active, E, K, lane, my_e,
              my_w);
  if (active && j < K) {
    topk_idx[(int64_t)t * K + j] = my_e;
    topk_w[(int64_t)t * K + j] = my_w;
    atomicOr(&s_mask[my_e], 1ull << tl);
  } else {
    my_e = -1;
  }
  __syncthreads();

  if (blk_hist != nullptr && tid < E)
    blk_hist[(int64_t)chunk * E + tid] = __popcll(s_mask[tid]);

  const int rank = my_e >= 0 ? __popcll(s_mask[my_e] & ((1ull << tl) - 1ull)) : -1;
  if (local_rank != nullptr && my_e >= 0) local_rank[(int64_t)t * K + j] = rank;

  if (single_chunk && offsets != nullptr) {
    if (wave == 0) {
      const int c = lane < E ? __popcll(s_mask[lane]) : 0;
      const int inc = wave_inclusive_scan(c);
      if (lane < E) {
        offsets[lane] = inc - c;
        s_off[lane] = inc - c;
        if (counts != nullptr) counts[lane] = c;
      }
      if (lane == 63) {
        offsets[E] = inc;
        for (int x = 1; x <= n_extra_groups; ++x) offsets[E + x] = inc + x * T;
      }
    }
    if (token_map != nullptr) {
      __syncthreads();
      if (my_e >= 0) {
        const int slot = s_off[my_e] + rank;
        token_map[slot] = t;
        if (slot_of != nullptr) slot_of[(int64_t)t * K + j] = slot;
      }
      // rows of the always-on groups: group E+x row t is token t
      const int S = T * K;
      for (int r = tid; r < n_extra_groups * T; r += blockDim.x) token_map[S + r] = r % T;
    }
  }
}

}  // namespace dsk
