// Linear maps of one to four token rows with fragment-tiled weights (the
// projections of an absorbed-MLA decode step), on the vector ALU:
//
//   out[b][m][n] = sum_k x[b][m][k] * w[b][n][k]      (fp32 sums, bf16 out)
//
// At one token a projection is a stream of its weights with two flops per
// weight element, so what matters is spreading that stream over the whole
// chip. The MFMA kernels need 32 weight rows and all of K per workgroup,
// which leaves a 2048-row projection with 64 workgroups. Here a group of
// lanes owns 8 rows: exactly one 128-byte line of each fragment half of the
// tiled layout (fragment (rb, ks) holds rows 32 rb .. 32 rb + 31 and K
// 16 ks .. 16 ks + 15; its first 256 elements are the K-half 0..7 of the 32
// rows, 8 per row). With 64 lanes per group (K >= 512) a 2048-row projection
// runs as 256 single-wave workgroups; with K < 512, 16 lanes per group and four
// groups per wave. Each lane sums its K slice with v_dot2_f32_bf16 in K order,
// the lanes of a group are added by a fixed DPP tree, so results are the same
// on every run.
#include "dsk_internal.hpp"
#include "gemm_common.hpp"
#include "route_token.hpp"

#include <algorithm>
#include <climits>

namespace dsk {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

struct RowsArgs {
  const uint16_t* x;
  int64_t ld_x, x_bs;      // token row stride, batch-entry stride (elements)
  const uint16_t* w;       // tiled [batch][N/32][K/16][64][8]
  int64_t w_bs;
  uint16_t* out0;          // outputs n < n_split
  int64_t ld_out0, out0_bs;
  uint16_t* out1;          // outputs n >= n_split, at column n - n_split
  int64_t ld_out1, out1_bs;
  int n_split, K, N;
};

constexpr int kRowsPerGroup = 8;  // one 128-byte line of a fragment half

// 8 bf16 products of w and x added to acc in order. The elements go through
// scalars first: hipcc (ROCm 7.2) compiles bit_cast(bf16x2, vector[e]) to
// element 0 for every e.
__device__ __forceinline__ float dot8(const u32x4_t& w, const u32x4_t& x, float acc) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t wq = w[q], xq = x[q];
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, wq),
                                          __builtin_bit_cast(bf16x2_t, xq), acc, false);
  }
  return acc;
}

template <int M, int LPR>
__global__ __launch_bounds__(64) void linear_rows_kernel(RowsArgs a) {
  constexpr int G = 64 / LPR;  // lane groups per wave
  // K chunks whose loads are issued together (a whole 2048-long row at 64 lanes)
  constexpr int kRowsBatch = LPR == 64 ? 4 : 1;
  const int lane = threadIdx.x;
  const int g = lane / LPR, li = lane % LPR;
  const int b = blockIdx.y;
  const int n0 = (blockIdx.x * G + g) * kRowsPerGroup;  // this group's first row
  const int nl = min(n0, a.N - kRowsPerGroup);          // rows past N: reload, unused
  const int rb = nl / 32, slab = (nl % 32) / kRowsPerGroup;
  const uint16_t* wb = a.w + b * a.w_bs + (int64_t)rb * (a.K / 16) * 512 + slab * 64;
  const uint16_t* xb = a.x + b * a.x_bs;
  const int nch = a.K / (8 * LPR);  // 8-element K chunks per lane

  float acc[M][kRowsPerGroup];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int i = 0; i < kRowsPerGroup; ++i) acc[m][i] = 0.f;

  for (int j0 = 0; j0 < nch; j0 += kRowsBatch) {
    u32x4_t wv[kRowsBatch][kRowsPerGroup], xv[kRowsBatch][M];
#pragma unroll
    for (int u = 0; u < kRowsBatch; ++u) {
      // chunk c = K elements 8c .. 8c+7: fragment c / 2, K half c % 2
      const int c = li + LPR * min(j0 + u, nch - 1);
      const uint16_t* wp = wb + (c >> 1) * 512 + (c & 1) * 256;
#pragma unroll
      for (int i = 0; i < kRowsPerGroup; ++i)
        wv[u][i] = *reinterpret_cast<const u32x4_t*>(wp + i * 8);
#pragma unroll
      for (int m = 0; m < M; ++m)
        xv[u][m] = *reinterpret_cast<const u32x4_t*>(xb + m * a.ld_x + c * 8);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the batch before the first use
#pragma unroll
    for (int u = 0; u < kRowsBatch; ++u) {
      if (j0 + u < nch) {
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
          for (int i = 0; i < kRowsPerGroup; ++i) acc[m][i] = dot8(wv[u][i], xv[u][m], acc[m][i]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // sums over the group's lanes (fixed DPP trees; every lane gets the total)
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int i = 0; i < kRowsPerGroup; ++i)
      acc[m][i] = LPR == 64 ? wave_sum(acc[m][i]) : row16_sum(acc[m][i]);

  // lane li of the group stores value idx = li + LPR * k: token idx / 8, row idx % 8
  if (n0 >= a.N) return;
#pragma unroll
  for (int k = 0; k * LPR < M * kRowsPerGroup; ++k) {
    const int idx = li + LPR * k;
    if (idx >= M * kRowsPerGroup) break;
    float v = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int i = 0; i < kRowsPerGroup; ++i)
        if (idx == m * kRowsPerGroup + i) v = acc[m][i];
    const int m = idx / kRowsPerGroup;
    const int n = n0 + idx % kRowsPerGroup;
    uint16_t* dst = n < a.n_split ? a.out0 + b * a.out0_bs + m * a.ld_out0 + n
                                  : a.out1 + b * a.out1_bs + m * a.ld_out1 + (n - a.n_split);
    *dst = f32_to_bf16(v);
  }
}

// -------------------------------------------------- routing + gate/up -------
// Routing and the first GEMM of a one-token MoE step in one launch: h[s] =
// silu(Wg x) * (Wu x) for the token's K experts (slot s: ascending expert) and the
// always-on groups (slot K + x). One wave per 8 gate rows and the matching 8 up rows of one
// group (a 64 KB unit at H = 2048); 1408 units over 256 CUs leave 6 on the fullest against
// 5.5 on average. A wave routes the token itself, in registers (route_token, on the gate's
// partial planes; the picks' bit mask gives the slot's expert), so nothing runs between the
// gate and this kernel, and the waves of the always-on groups, which need no routing,
// stream meanwhile. Workgroup 0 stores the routing for the kernels after it.
//
// A lane holds one row and every eighth chunk, so each load instruction covers eight whole
// lines and the weights pass the caches once. (With a line per lane and its 8 rows in 8
// instructions, as linear_rows_kernel reads them, a CU holds more lines than its L1 and
// fetches them again: 26 us, and 55 with loads that bypass the caches.) Against the MFMA
// kernel of small groups with the routing in its prologue, which this replaces at one
// token: 22.2 -> 18.8 us; the layer, with the next kernel's reads in the same order,
// 36.6 -> 31.6 us.
// Lane (r8, c8)'s first 16 bytes of row n0 + r8 (n0 a multiple of 8) of a [N, K] weight:
// chunk c8 of the row's 8-element chunks.
template <bool TILED>
__device__ __forceinline__ const uint16_t* slab_lane(const uint16_t* w, int K, int n0, int r8,
                                                     int c8) {
  if constexpr (TILED)
    return w + (int64_t)(n0 / 32) * (K / 16) * 512 + (n0 % 32 + r8) * 8 + (c8 >> 1) * 512 +
           (c8 & 1) * 256;
  else
    return w + (int64_t)(n0 + r8) * K + c8 * 8;
}

// Sum over the 8 lanes that hold one row (lanes 8 apart), in a fixed order; all get it.
__device__ __forceinline__ float chunk_lanes_sum(float v) {
  v += __shfl_xor(v, 8, 64);
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}

struct TokenGemm1Args {
  const float* parts;  // [n_parts][E] partial gate sums
  int n_parts;
  int64_t part_stride;
  const float* bias;
  const uint16_t* x;   // [H]
  const uint16_t* w1;  // [E + nsh, 2 I, H], row-major or tiled
  uint16_t* h;         // [K + nsh, I]
  int E, K, nsh, H, I;
  int32_t* idx;
  float* w;
  int32_t* counts;
  int32_t* offsets;
  int32_t* token_map;
  int32_t* slot_of;
};

template <bool TILED>
__global__ __launch_bounds__(64) void token_gemm1_kernel(TokenGemm1Args a) {
  constexpr int kBatch = 8;  // steps of 64 K elements in flight: 16 KB of weights
  const int lane = threadIdx.x;
  const int units = a.I / kRowsPerGroup;
  const int slot = blockIdx.x / units, n0 = (blockIdx.x - slot * units) * kRowsPerGroup;
  int g = a.E + slot - a.K;
  if (slot < a.K) {  // uniform
    int my_e;
    float my_w;
    // every 16-lane row of the wave routes the same token
    route_token(a.parts, a.E, a.n_parts, a.part_stride, a.bias, 0, true, true, a.E, a.K, lane,
                my_e, my_w);
    uint64_t mask = 0;
    for (int k = 0; k < a.K; ++k) mask |= 1ull << (__builtin_amdgcn_readlane(my_e, k) & 63);
    uint64_t rest = mask;
    for (int k = 0; k < slot; ++k) rest &= rest - 1;
    g = __ffsll((unsigned long long)rest) - 1;
    if (blockIdx.x == 0) {
      if (lane < a.K) {
        a.idx[lane] = my_e;
        a.w[lane] = my_w;
        a.slot_of[lane] = __popcll(mask & ((1ull << (my_e & 63)) - 1ull));
      }
      if (lane < a.E) {
        a.offsets[lane] = __popcll(mask & ((1ull << lane) - 1ull));
        a.counts[lane] = (int)((mask >> lane) & 1);
      }
      for (int i = lane; i <= a.nsh; i += 64) a.offsets[a.E + i] = a.K + i;
      for (int i = lane; i < a.K + a.nsh; i += 64) a.token_map[i] = 0;
    }
  }
  // lane = (row lane % 8, chunk lane / 8 of each step's 8): a load instruction covers eight
  // whole 128-byte lines in either layout
  const int r8 = lane & 7, c8 = lane >> 3;
  const int steps = a.H / 64;
  const uint16_t* base = a.w1 + (int64_t)g * 2 * a.I * a.H;
  const uint16_t* gate = slab_lane<TILED>(base, a.H, n0, r8, c8);
  const uint16_t* up = slab_lane<TILED>(base, a.H, a.I + n0, r8, c8);
  const uint16_t* x = a.x + c8 * 8;
  constexpr int kStep = TILED ? 2048 : 64;  // elements per 8 chunks
  float ag = 0.f, au = 0.f;
  for (int j0 = 0; j0 < steps; j0 += kBatch) {
    u32x4_t wg[kBatch], wu[kBatch], xv[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int j = min(j0 + u, steps - 1);  // past the row: reload, unused
      wg[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(gate + j * kStep));
      wu[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(up + j * kStep));
      xv[u] = *reinterpret_cast<const u32x4_t*>(x + j * 64);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the batch before the first use
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (j0 + u < steps) {
        ag = dot8(wg[u], xv[u], ag);
        au = dot8(wu[u], xv[u], au);
      }
    }
  }
  ag = chunk_lanes_sum(ag);
  au = chunk_lanes_sum(au);
  if (c8 == 0) a.h[(int64_t)slot * a.I + n0 + r8] = f32_to_bf16(silu_f(ag) * au);
}

int launch_token_gemm1(const float* parts, int n_parts, int64_t part_stride, const float* bias,
                       const uint16_t* x, const uint16_t* w1, bool tiled, uint16_t* h, int E,
                       int K, int nsh, int H, int I, int32_t* idx, float* w, int32_t* counts,
                       int32_t* offsets, int32_t* token_map, int32_t* slot_of, hipStream_t st) {
  DSK_REQUIRE(n_parts >= 1 && n_parts <= kMaxGateParts && E >= 1 && E <= 64 && K >= 1 &&
                  K <= std::min(E, 16) && nsh >= 0 && H % 64 == 0 && I % 32 == 0,
              DSK_ERR_INVALID_ARG, "token_gemm1: sizes out of range");
  const TokenGemm1Args a{parts, n_parts, part_stride, bias, x, w1, h, E, K, nsh, H, I,
                         idx, w, counts, offsets, token_map, slot_of};
  const dim3 grid((unsigned)((K + nsh) * (I / kRowsPerGroup)));
  if (tiled)
    hipLaunchKernelGGL(token_gemm1_kernel<true>, grid, dim3(64), 0, st, a);
  else
    hipLaunchKernelGGL(token_gemm1_kernel<false>, grid, dim3(64), 0, st, a);
  return check_launch("token_gemm1_kernel");
}

// ------------------------------------------- down projection + combine ----
// The MoE layer's second GEMM and its combine in one launch, for the smallest steps:
//
//   out[t][n] = sum_k wt[t][k] * y[slot_of[t][k]][n] + sum_x y[S + x T + t][n],
//   y[s][n] = bf16(sum_i h[s][i] * w2[g(s)][n][i])
//
// with the rounding of y and the order of the sum (slots ascending, then the always-on
// groups, fp32, one rounding) of combine_slots_kernel.
//
// At one token the GEMM streams 46 MB for 12 us and the combine that follows costs a launch
// (4.6 us) for 32 KB. Both are one launch if a workgroup has the same columns of every
// busy group, and the even split of the columns also gives each CU the same bytes: a
// workgroup owns 8 columns (one 128-byte line of each fragment half, as above), each of its
// 8 waves takes every eighth busy group, 11 KB of its rows in flight at once, and the rows
// of y meet in LDS. The layer at one token 39.0 -> 36.6 us by this launch alone (with a line
// per lane), at two tokens with 9 busy groups 49 -> 43 and with 13 58 -> 55. From three
// tokens up a wave's bursts over several groups no longer fill the CU's queue (three tokens
// 75 -> 77 us, four 80 -> 86), so larger steps keep the two launches.
constexpr int kCombineWavesG2 = 8;
constexpr int kCombineCols = 8;
constexpr int kG2Batch = 11;   // steps of 64 K elements in flight (1408 = 22 x 64)
constexpr int kG2MaxSlots = 256;
constexpr int kG2MaxK = 8;

struct Gemm2CombineArgs {
  const uint16_t* h;  // [slots, I]
  const uint16_t* w2; // [G, H, I], row-major or tiled
  const int32_t* offsets;  // [G + 1]
  const int32_t* slot_of;  // [T, K]
  const float* topk_w;     // [T, K]
  uint16_t* out;           // [T, H]
  int T, K, G, nsh, H, I, slots;
};

template <int MT, bool TILED>
__global__ __launch_bounds__(64 * kCombineWavesG2) void gemm2_combine_kernel(Gemm2CombineArgs a) {
  __shared__ __attribute__((aligned(16))) float s_y[kG2MaxSlots][kCombineCols];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * kCombineCols;
  const int r8 = lane & 7, c8 = lane >> 3;  // row and chunk of a lane, as above
  const int steps = a.I / 64;
  constexpr int kStep = TILED ? 2048 : 64;

  // busy groups, lane = group (G <= 128: two halves)
  int lo0 = 0, hi0 = 0, lo1 = 0, hi1 = 0;
  if (lane < a.G) {
    lo0 = min(max(a.offsets[lane], 0), a.slots);
    hi0 = min(max(a.offsets[lane + 1], lo0), a.slots);
  }
  if (lane + 64 < a.G) {
    lo1 = min(max(a.offsets[lane + 64], 0), a.slots);
    hi1 = min(max(a.offsets[lane + 65], lo1), a.slots);
  }
  // the combine's slots and weights of token tid / 8, in ascending slot order, while the
  // weights stream
  const int t = tid / kCombineCols, col = tid % kCombineCols;
  int s[kG2MaxK];
  float wt[kG2MaxK];
#pragma unroll
  for (int k = 0; k < kG2MaxK; ++k) {
    const bool on = t < a.T && k < a.K;
    const int sk = on ? a.slot_of[t * a.K + k] : -1;
    s[k] = sk >= 0 && sk < a.slots ? sk : INT_MAX;
    wt[k] = on ? a.topk_w[t * a.K + k] : 0.f;
  }
  const uint64_t m0 = __ballot(hi0 > lo0), m1 = __ballot(hi1 > lo1);
  const int c0 = __popcll(m0), busy = c0 + __popcll(m1);

  for (int ord = wave; ord < busy; ord += kCombineWavesG2) {
    // the ord-th busy group
    const bool upper = ord >= c0;
    const uint64_t mask = upper ? m1 : m0;
    const int want = upper ? ord - c0 : ord;
    const bool mine = ((mask >> lane) & 1) && __popcll(mask & ((1ull << lane) - 1ull)) == want;
    const int src = __ffsll((unsigned long long)__ballot(mine)) - 1;
    const int g = src + (upper ? 64 : 0);
    const int lo = __builtin_amdgcn_readlane(upper ? lo1 : lo0, src);
    const int rows = min(__builtin_amdgcn_readlane(upper ? hi1 : hi0, src) - lo, MT);
    const uint16_t* wb = slab_lane<TILED>(a.w2 + (int64_t)g * a.H * a.I, a.I, n0, r8, c8);
    const uint16_t* hb = a.h + (int64_t)lo * a.I + c8 * 8;
    float acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = 0.f;
    for (int j0 = 0; j0 < steps; j0 += kG2Batch) {
      u32x4_t wv[kG2Batch], xv[kG2Batch][MT];
#pragma unroll
      for (int u = 0; u < kG2Batch; ++u) {
        const int j = min(j0 + u, steps - 1);  // past the row: reload, unused
        wv[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wb + j * kStep));
#pragma unroll
        for (int m = 0; m < MT; ++m)
          xv[u][m] = *reinterpret_cast<const u32x4_t*>(hb + (int64_t)min(m, rows - 1) * a.I + j * 64);
      }
      __builtin_amdgcn_sched_barrier(0);  // every load of the batch before the first use
#pragma unroll
      for (int u = 0; u < kG2Batch; ++u) {
        if (j0 + u < steps) {
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m] = dot8(wv[u], xv[u][m], acc[m]);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float v = bf16_to_f32(f32_to_bf16(chunk_lanes_sum(acc[m])));
      if (m < rows && c8 == 0) s_y[lo + m][r8] = v;
    }
  }
  // fixed sorting network on compile-time indices
#pragma unroll
  for (int x = 0; x < kG2MaxK; ++x) {
#pragma unroll
    for (int y = 0; y < kG2MaxK - 1 - x; ++y) {
      if (s[y] > s[y + 1]) {
        const int ts = s[y]; s[y] = s[y + 1]; s[y + 1] = ts;
        const float tw = wt[y]; wt[y] = wt[y + 1]; wt[y + 1] = tw;
      }
    }
  }
  __syncthreads();
  if (t >= a.T) return;
  float o = 0.f;
#pragma unroll
  for (int k = 0; k < kG2MaxK; ++k)
    if (s[k] != INT_MAX) o = fmaf(wt[k], s_y[s[k]][col], o);
  for (int x = 0; x < a.nsh; ++x) o += s_y[a.T * a.K + x * a.T + t][col];
  a.out[(int64_t)t * a.H + n0 + col] = f32_to_bf16(o);
}

bool gemm2_combine_takes(int T, int K, int G, int nsh, int H, int I) {
  return T >= 1 && T <= kGemm2CombineTokens && K <= kG2MaxK && G <= 128 &&
         T * (K + nsh) <= kG2MaxSlots && H % 32 == 0 && I % 64 == 0;
}

int launch_gemm2_combine(const uint16_t* h, const uint16_t* w2, bool tiled,
                         const int32_t* offsets, const int32_t* slot_of, const float* topk_w,
                         uint16_t* out, int T, int K, int G, int nsh, int H, int I,
                         hipStream_t st) {
  DSK_REQUIRE(gemm2_combine_takes(T, K, G, nsh, H, I), DSK_ERR_INVALID_ARG,
              "gemm2_combine: sizes out of range");
  const Gemm2CombineArgs a{h, w2, offsets, slot_of, topk_w, out, T, K, G, nsh, H, I,
                           T * (K + nsh)};
  const dim3 grid((unsigned)(H / kCombineCols));
  static_assert(kGemm2CombineTokens == 2, "a variant per token count");
  auto kern = T == 1 ? (tiled ? gemm2_combine_kernel<1, true> : gemm2_combine_kernel<1, false>)
                     : (tiled ? gemm2_combine_kernel<2, true> : gemm2_combine_kernel<2, false>);
  hipLaunchKernelGGL(kern, grid, dim3(64 * kCombineWavesG2), 0, st, a);
  return check_launch("gemm2_combine_kernel");
}

template <int LPR>
static void launch_rows_lpr(const RowsArgs& a, int M, int batch, hipStream_t st) {
  constexpr int G = 64 / LPR;
  const dim3 grid((unsigned)((a.N + kRowsPerGroup * G - 1) / (kRowsPerGroup * G)),
                  (unsigned)batch);
  switch (M) {
    case 1: hipLaunchKernelGGL((linear_rows_kernel<1, LPR>), grid, dim3(64), 0, st, a); break;
    case 2: hipLaunchKernelGGL((linear_rows_kernel<2, LPR>), grid, dim3(64), 0, st, a); break;
    case 3: hipLaunchKernelGGL((linear_rows_kernel<3, LPR>), grid, dim3(64), 0, st, a); break;
    default: hipLaunchKernelGGL((linear_rows_kernel<4, LPR>), grid, dim3(64), 0, st, a); break;
  }
}

}  // namespace dsk

using namespace dsk;

extern "C" int dsk_linear_rows(const dsk_bf16* x, int64_t ld_x, int64_t x_batch_stride,
                               const dsk_bf16* w_tiled, int64_t w_batch_stride, dsk_bf16* out0,
                               int64_t ld_out0, int64_t out0_batch_stride, dsk_bf16* out1,
                               int64_t ld_out1, int64_t out1_batch_stride, int n_split,
                               int batch, int M, int K, int N, void* stream) {
  DSK_REQUIRE(batch >= 0 && M >= 0 && K > 0 && N > 0, DSK_ERR_INVALID_ARG,
              "linear_rows: invalid sizes");
  DSK_REQUIRE(M <= 4, DSK_ERR_INVALID_ARG, "linear_rows: at most 4 token rows");
  DSK_REQUIRE(K % 128 == 0 && N % 32 == 0, DSK_ERR_INVALID_ARG,
              "linear_rows: K must be a multiple of 128 and N of 32 (tiled weight)");
  DSK_REQUIRE(n_split >= 0 && n_split <= N, DSK_ERR_INVALID_ARG,
              "linear_rows: n_split must be in [0, N]");
  if (batch == 0 || M == 0) return DSK_OK;
  DSK_REQUIRE(x && w_tiled && (n_split == 0 || out0) && (n_split == N || out1),
              DSK_ERR_NULL_PTR, "linear_rows: NULL pointer");
  DSK_REQUIRE(aligned16(x) && aligned16(w_tiled) && ld_x % 8 == 0 && x_batch_stride % 8 == 0 &&
                  w_batch_stride % 8 == 0,
              DSK_ERR_ALIGNMENT, "linear_rows: x rows and weights must be 16-byte aligned");
  DSK_REQUIRE(ld_x >= K && (n_split == 0 || ld_out0 >= n_split) &&
                  (n_split == N || ld_out1 >= N - n_split),
              DSK_ERR_INVALID_ARG, "linear_rows: row stride smaller than the row");
  DSK_REQUIRE(batch <= 65535, DSK_ERR_INVALID_ARG, "linear_rows: batch must be at most 65535");
  RowsArgs a{reinterpret_cast<const uint16_t*>(x), ld_x, x_batch_stride,
             reinterpret_cast<const uint16_t*>(w_tiled), w_batch_stride,
             reinterpret_cast<uint16_t*>(out0), ld_out0, out0_batch_stride,
             reinterpret_cast<uint16_t*>(out1), ld_out1, out1_batch_stride, n_split, K, N};
  if (K % 512 == 0) launch_rows_lpr<64>(a, M, batch, as_stream(stream));
  else launch_rows_lpr<16>(a, M, batch, as_stream(stream));
  return check_launch("linear_rows_kernel");
}
