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
// 8 waves takes every eighth busy group, all weight loads of a 1408-long row in flight at
// once, and the rows of y meet in LDS. The layer at one token 39.0 -> 36.6 us, at two
// tokens with 9 busy groups 49 -> 44 and with 13 58 -> 58. From three tokens up a wave's
// bursts over several groups no longer fill the CU's queue (three tokens with 17 to 19 busy
// groups 76 -> 79 us, four 82 -> 93), so larger steps keep the two launches.
constexpr int kCombineWavesG2 = 8;
constexpr int kCombineCols = 8;
constexpr int kG2Batch = 3;    // 8-element K chunks per lane in flight (1408 = 2.75 x 512)
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
  const int nch = a.I / 8;

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
    const uint16_t* wb = a.w2 + (int64_t)g * a.H * a.I;
    wb += TILED ? (int64_t)(n0 / 32) * (a.I / 16) * 512 + (n0 % 32 / kCombineCols) * 64
                : (int64_t)n0 * a.I;
    float acc[MT][kCombineCols];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < kCombineCols; ++i) acc[m][i] = 0.f;
    for (int j0 = 0; j0 < nch; j0 += 64 * kG2Batch) {
      u32x4_t wv[kG2Batch][kCombineCols], xv[kG2Batch][MT];
#pragma unroll
      for (int u = 0; u < kG2Batch; ++u) {
        const int c = min(j0 + 64 * u + lane, nch - 1);  // past the row: reload, unused
        const uint16_t* wp = TILED ? wb + (c >> 1) * 512 + (c & 1) * 256 : wb + c * 8;
#pragma unroll
        for (int i = 0; i < kCombineCols; ++i)
          wv[u][i] = *reinterpret_cast<const u32x4_t*>(wp + (int64_t)i * (TILED ? 8 : a.I));
#pragma unroll
        for (int m = 0; m < MT; ++m)
          xv[u][m] = *reinterpret_cast<const u32x4_t*>(a.h + (int64_t)(lo + min(m, rows - 1)) * a.I +
                                                       c * 8);
      }
      __builtin_amdgcn_sched_barrier(0);  // every load of the batch before the first use
#pragma unroll
      for (int u = 0; u < kG2Batch; ++u) {
        if (j0 + 64 * u + lane < nch) {
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < kCombineCols; ++i)
              acc[m][i] = dot8(wv[u][i], xv[u][m], acc[m][i]);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < rows) {  // uniform
        float v[kCombineCols];
#pragma unroll
        for (int i = 0; i < kCombineCols; ++i) v[i] = bf16_to_f32(f32_to_bf16(wave_sum(acc[m][i])));
        if (lane == 0) {
#pragma unroll
          for (int i = 0; i < kCombineCols; ++i) s_y[lo + m][i] = v[i];
        }
      }
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
         T * (K + nsh) <= kG2MaxSlots && H % 32 == 0 && I % 16 == 0;
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
