// Grouped GEMM for medium problems (gfx950): tiles of 64 or 128 token rows, two or
// more workgroups per CU. It runs the shapes that lie between the weight-streaming
// kernel (groups of at most 64 rows) and the 256 x 256 tile kernels (several rounds
// of full tiles): the expert GEMMs of a few hundred tokens, where a 256-row tile is
// mostly padding, and dense projections whose 256 x 256 tiles do not cover the CUs.
//
// Data path, as in the one-wave-per-SIMD kernel (gemm.hip): a wave owns TN blocks of
// 32 weight rows against every token row of the tile. Fragment-tiled weights go from
// memory straight into registers, two stages of 64 K ahead (nobody else needs them);
// the token rows go through a 4-deep LDS ring filled by global->LDS DMA three stages
// ahead and are read back by all 4 waves. Row-major weights go through the ring beside
// the tokens (a fragment load would touch 32 rows for 32 bytes each; the DMA moves
// whole 128-byte lines). One barrier per stage. A workgroup runs one tile; several
// share a CU, so one's prologue, epilogue and waits are covered by another's loads and
// MFMAs, without a persistent stage stream.
//
// The order of memory operations per stage is fixed (the DMA instructions, then with
// tiled weights TN weight loads per K step), which the explicit vmcnt waits count on;
// past the end of K the last stage is repeated into slots and registers that nobody
// reads again.
#include "dsk_internal.hpp"
#include "gemm_common.hpp"
#include "gemm_sched.hpp"

#include <type_traits>

namespace dsk {

constexpr int kMidWaves = 4;
constexpr int kMidThreads = 64 * kMidWaves;
constexpr int kMidBK = 64;

template <int TM, int TN, bool SWIGLU, bool GATHER, bool TILED>
struct MidCfg {
  static_assert(TM == 2 || TM == 4, "64 or 128 token rows per tile");
  static_assert(TN == 1 || TN == 2, "one or two weight blocks per wave");
  static_assert(!SWIGLU || (TILED ? TN == 2 : TN == 1),
                "SwiGLU pairs a gate and an up block (tiled) or the halves of one block");
  static constexpr int BM = 32 * TM;
  static constexpr int BN = 32 * TN * kMidWaves;  // weight rows
  static constexpr int OUT_N = SWIGLU ? BN / 2 : BN;
  static constexpr int kStageBytes = (BM + (TILED ? 0 : BN)) * kMidBK * 2;
  // row-major weights: what leaves two workgroups per CU
  static constexpr int kRing = TILED ? 4 : 3 * kStageBytes <= 76 * 1024 ? 3 : 2;
};

// One tile W of the launch; s_inc / s_mb / s_me: the group table.
template <int TM, int TN, bool SWIGLU, bool GATHER, bool TILED>
__device__ __forceinline__ void mid_tile(const GemmArgs& p, int W, int NT, char* s_ring,
                                         const int* s_inc, const int* s_mb, const int* s_me) {
  using Cfg = MidCfg<TM, TN, SWIGLU, GATHER, TILED>;
  constexpr int BM = Cfg::BM, OUT_N = Cfg::OUT_N, RING = Cfg::kRing;
  constexpr int KSTEPS = kMidBK / 16;
  constexpr int kStageBytes = Cfg::kStageBytes;
  constexpr int W_INSTS = TILED ? 0 : 4 * TN;  // weight DMA instructions per wave per stage
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- the tile: group g, rows [m0, me), output columns from n0
  int g = 0, mb = 0, gme = p.M, local = W;
  if (p.offsets != nullptr) {
    int lo = 0, hi = p.G - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_inc[mid] > W) hi = mid; else lo = mid + 1;
    }
    g = __builtin_amdgcn_readfirstlane(lo);
    local = W - (g > 0 ? s_inc[g - 1] : 0);
    mb = s_mb[g];
    gme = s_me[g];
  }
  const int mt = (gme - mb + BM - 1) / BM;
  const int nblk = (gme - mb + 31) / 32;
  int nt, mi;
  sched_group_tile(local, mt, NT, &nt, &mi);
  // the even split of the blocks; the product fits 32 bits up to kMidMaxRows (sched_tile_block
  // holds for any count, at 0.1-0.2 us a launch)
  nt = __builtin_amdgcn_readfirstlane(nt);
  const int m0 = __builtin_amdgcn_readfirstlane(mb + 32 * (mi * nblk / mt));
  const int me = __builtin_amdgcn_readfirstlane(min(mb + 32 * ((mi + 1) * nblk / mt), gme));
  const int n0 = nt * OUT_N;
  const int tma = (me - m0 + 31) / 32;  // token blocks with rows
  const int nk = p.K / kMidBK;

  // DMA: instruction i of a wave moves rows 8 (wave + 4 i) .. + 7 of the tile's token
  // (or weight) rows, 128 bytes each, chunk-swizzled
  const int dma_row = lane >> 3;
  const int dma_chunk = (lane & 7) ^ dma_row ^ (wave & 1);

  // ---- weights: byte offset of this wave's block j at k = 0 (tiled), or of the row
  // that its DMA instruction i moves
  const char* Bg = reinterpret_cast<const char*>(p.B + (int64_t)g * p.b_group_stride);
  uint32_t b_off[TILED ? TN : W_INSTS];
  if constexpr (TILED) {
    const int last = p.N / 32 - 1;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      int rb;
      if constexpr (SWIGLU) {
        const int ob = min(n0 / 32 + wave, last);
        rb = j == 0 ? ob : p.up_row_offset / 32 + ob;  // gate rows, then up rows
      } else {
        rb = min(n0 / 32 + TN * wave + j, last);
      }
      b_off[j] = (uint32_t)((((int64_t)rb * (p.K / 16)) * 512 + lane * 8) * 2);
    }
  } else {
#pragma unroll
    for (int i = 0; i < W_INSTS; ++i) {
      const int r = 8 * (wave + kMidWaves * i) + dma_row;
      int row;
      if constexpr (SWIGLU) {  // a wave's block: 16 gate rows, then the 16 matching up rows
        const int col = min(n0 + 16 * (r >> 5) + (r & 15), p.N - 1);
        row = (r & 16) ? p.up_row_offset + col : col;
      } else {
        row = min(n0 + r, p.N - 1);
      }
      b_off[i] = (uint32_t)(((int64_t)row * p.ldb + dma_chunk * 8) * 2);
    }
  }
  auto issue_b = [&](bf16x8_t (&dst)[TN], int stage, int k) __attribute__((always_inline)) {
    if constexpr (TILED) {
      const uint32_t koff = (uint32_t)(min(stage, nk - 1) * KSTEPS + k) * 1024;
#pragma unroll
      for (int j = 0; j < TN; ++j)
        dst[j] = *reinterpret_cast<const bf16x8_t*>(Bg + (b_off[j] + koff));
    }
  };

  // ---- tokens: rows past the tile repeat its first row
  const char* Abase = reinterpret_cast<const char*>(p.A);
  const int row_limit = GATHER ? p.a_rows_limit : p.M;
  uint32_t a_off[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + 8 * (wave + kMidWaves * i) + dma_row;
    int row = m < me ? m : m0;
    if constexpr (GATHER) row = p.a_rows[row];
    row = (row >= 0 && row < row_limit) ? row : 0;
    a_off[i] = (uint32_t)(((int64_t)row * p.lda + dma_chunk * 8) * 2);
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(s_ring));
  auto issue_dma = [&](int stage) __attribute__((always_inline)) {
    const uint32_t koff = (uint32_t)min(stage, nk - 1) * kMidBK * 2;
    const uint32_t dst = lds_base + (stage % RING) * kStageBytes;
#pragma unroll
    for (int i = 0; i < W_INSTS; ++i)
      dma_1kb(Bg, b_off[i] + koff, dst + BM * 128 + (wave + kMidWaves * i) * 1024);
#pragma unroll
    for (int i = 0; i < TM; ++i)
      dma_1kb(Abase, a_off[i] + koff, dst + (wave + kMidWaves * i) * 1024);
  };

  // weight fragments: register set = stage parity (tiled) or K step parity (from the LDS)
  bf16x8_t fb[2][TILED ? KSTEPS : 1][TN];
  bf16x8_t fa[2][TM];          // token fragments, double-buffered by K step
  floatx16_t acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.f;
  const u32x4_t* lds4 = reinterpret_cast<const u32x4_t*>(s_ring);
  auto read_frags = [&](int set, int slot, int kk) __attribute__((always_inline)) {
    const u32x4_t* As = lds4 + slot * (kStageBytes / 16);
    const int ch = 2 * kk + (lane >> 5);
    if constexpr (!TILED) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[set][0][j] = __builtin_bit_cast(
            bf16x8_t, As[BM * 8 + lds_swz<8>(32 * (TN * wave + j) + (lane & 31), ch)]);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[set][i] = __builtin_bit_cast(bf16x8_t, As[lds_swz<8>(32 * i + (lane & 31), ch)]);
  };

  // ---- prologue: the ring's first stages in flight (tiled: A0 B0 A1 B1 A2), stage 0
  // landed
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) {
    issue_dma(s);
    if (TILED && s < 2) {
#pragma unroll
      for (int k = 0; k < KSTEPS; ++k) issue_b(fb[s][k], s, k);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // what follows stage 0's DMA: B0 A1 B1 A2, or the other stages' DMA
  wait_vmcnt<TILED ? 2 * TM + 2 * KSTEPS * TN : (RING - 2) * (TM + W_INSTS)>();
  lds_barrier();
  read_frags(0, 0, 0);

  auto stage = [&](auto set_c, int s) __attribute__((always_inline)) {
    constexpr int SET = decltype(set_c)::value;
    issue_dma(s + RING - 1);  // into the slot of stage s - 1, which every wave has read
#pragma unroll
    for (int k = 0; k < KSTEPS; ++k) {
      if (k == KSTEPS - 1) {
        // Stage s + 1 has landed. Tiled: after A(s + 1) came at least B(s) or B(s + 1)
        // (4 TN), A(s + 2), A(s + 3) and 3 TN loads of B(s + 2). Row-major: the DMA of
        // the RING - 2 stages after it.
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<TILED ? 2 * TM + 7 * TN : (RING - 2) * (TM + W_INSTS)>();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): own LDS reads done
        lds_barrier();
        read_frags((k + 1) & 1, (s + 1) % RING, 0);
      } else {
        read_frags((k + 1) & 1, s % RING, k + 1);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i < TM / 2 || i < tma) {  // uniform
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                TILED ? fb[SET][k][j] : fb[k & 1][0][j], fa[k & 1][i], acc[j][i], 0, 0, 0);
        }
      }
      issue_b(fb[SET][TILED ? k : 0], s + 2, k);
    }
  };
#pragma unroll 1
  for (int s = 0; s < nk; s += 2) {
    stage(std::integral_constant<int, 0>{}, s);
    if (s + 1 < nk) stage(std::integral_constant<int, 1>{}, s + 1);
  }

  // ---- epilogue through the LDS: each wave stages one 32-row block at a time and
  // stores whole row segments (32, 64 or 128 bytes)
  wait_vmcnt<0>();  // no DMA lands in the ring any more
  __builtin_amdgcn_s_waitcnt(0xC07F);
  lds_barrier();
  constexpr bool kHalves = SWIGLU && TN == 1;  // gate and up rows in one block
  constexpr int JN = SWIGLU ? 1 : TN;
  constexpr int QG = kHalves ? 2 : 4;          // groups of 8 output columns per block
  constexpr int ROW_BYTES = 16 * QG * JN;
  constexpr int CHUNKS = ROW_BYTES / 16;
  constexpr int ROWS_PER_INST = 64 / CHUNKS;
  auto swz = [](int row) {
    return CHUNKS == 2 ? (row >> 3) & 1 : CHUNKS == 4 ? (row >> 2) & 3 : (row >> 1) & 7;
  };
  char* st = s_ring + wave * 4096;
  const int r32 = lane & 31, h = lane >> 5;
  const int col0 = n0 + 8 * QG * JN * wave;
  const int rl = lane / CHUNKS, cl = lane % CHUNKS;
  // row statistics (GemmArgs): whole 256-column tiles, TN = 2 only
  constexpr bool kRowOps = !SWIGLU && !GATHER && TILED && TN == 2;
  const bool scale_rows = kRowOps && p.rowscale_ss != nullptr;
  const bool sum_rows = kRowOps && p.rowsq_out != nullptr && n0 >= p.rowsq_c0 && n0 < p.rowsq_c1;
  float* s_ss = reinterpret_cast<float*>(s_ring + kMidWaves * 4096);  // [wave][row of the tile]
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (i >= tma) continue;
    float rs = 1.f;
    if constexpr (kRowOps) {
      if (scale_rows) {
        const int m = min(m0 + 32 * i + r32, p.M - 1);
        float ss = p.rowscale_ss[m];
        for (int q = 1; q < p.rowscale_parts; ++q) ss += p.rowscale_ss[q * p.ld_rowscale + m];
        rs = rsqrtf(ss * (1.f / p.rowscale_cols) + p.rowscale_eps);
      }
    }
#pragma unroll
    for (int j = 0; j < JN; ++j) {
#pragma unroll
      for (int qg = 0; qg < QG; ++qg) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if constexpr (kHalves) v[c] = silu_f(acc[0][i][4 * qg + c]) * acc[0][i][8 + 4 * qg + c];
          else if constexpr (SWIGLU) v[c] = silu_f(acc[0][i][4 * qg + c]) * acc[1][i][4 * qg + c];
          else if constexpr (kRowOps) v[c] = acc[j][i][4 * qg + c] * rs;
          else v[c] = acc[j][i][4 * qg + c];
        }
        u32x2_t o;
        o[0] = pack_bf16x2(v[0], v[1]);
        o[1] = pack_bf16x2(v[2], v[3]);
        const int ch = 4 * j + qg;
        *reinterpret_cast<u32x2_t*>(st + r32 * ROW_BYTES + ((ch ^ swz(r32)) * 16) +
                                    ((h ^ ((r32 >> 4) & 1)) * 8)) = o;
      }
    }
#pragma unroll
    for (int q = 0; q < 32 / ROWS_PER_INST; ++q) {
      const int rr = q * ROWS_PER_INST + rl;
      u32x4_t d = *reinterpret_cast<const u32x4_t*>(st + rr * ROW_BYTES + ((cl ^ swz(rr)) * 16));
      if ((rr >> 4) & 1) d = u32x4_t{d[2], d[3], d[0], d[1]};  // halves were swapped
      const int m = m0 + 32 * i + rr;
      const int col = col0 + 8 * cl;
      if (m < me && col < p.N) *reinterpret_cast<u32x4_t*>(p.C + (int64_t)m * p.ldc + col) = d;
      if constexpr (kRowOps) {
        if (sum_rows) {
          // squares of the stored (bf16) values, summed over the row's 8 lanes
          // (quad swaps, then the half-row mirror)
          float sq = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float lo = bf16lo(d[e]), hi = bf16hi(d[e]);
            sq = fmaf(lo, lo, sq);
            sq = fmaf(hi, hi, sq);
          }
          sq += dpp_f32<0xB1>(0.f, sq);
          sq += dpp_f32<0x4E>(0.f, sq);
          sq += dpp_f32<0x141>(0.f, sq);
          if (cl == 0) s_ss[wave * BM + 32 * i + rr] = sq;
        }
      }
    }
  }
  if constexpr (kRowOps) {
    if (sum_rows) {
      __syncthreads();
      // the tile's row sums, the four waves' column ranges added in order
      if (tid < 32 * tma && m0 + tid < me) {
        const float ss = ((s_ss[tid] + s_ss[BM + tid]) + s_ss[2 * BM + tid]) + s_ss[3 * BM + tid];
        p.rowsq_out[(int64_t)((n0 - p.rowsq_c0) / OUT_N) * p.ld_rowsq + m0 + tid] = ss;
      }
    }
  }
}

template <int TM, int TN, bool SWIGLU, bool GATHER, bool TILED>
__global__ __launch_bounds__(kMidThreads, 2) void mid_gemm_kernel(GemmArgs p, int chunk) {
  using Cfg = MidCfg<TM, TN, SWIGLU, GATHER, TILED>;
  constexpr int BM = Cfg::BM;
  __shared__ __attribute__((aligned(1024))) char s_ring[Cfg::kRing * Cfg::kStageBytes];
  __shared__ int s_inc[kMaxGroups];
  __shared__ int s_mb[kMaxGroups];
  __shared__ int s_me[kMaxGroups];
  const int tid = threadIdx.x;
  const int NT = (p.N + Cfg::OUT_N - 1) / Cfg::OUT_N;
  // ---- group table: row ranges and inclusive prefix of tile counts
  int total = (p.M + BM - 1) / BM * NT;
  if (p.offsets != nullptr) {
    if (tid < kMaxGroups) {
      int cnt = 0;
      if (tid < p.G) {
        const int lo = min(max(p.offsets[tid], 0), p.M);
        const int hi = min(max(p.offsets[tid + 1], lo), p.M);
        s_mb[tid] = lo;
        s_me[tid] = hi;
        cnt = ((hi - lo + BM - 1) / BM) * NT;
      }
      s_inc[tid] = wave_inclusive_scan(cnt);
    }
    __syncthreads();
    const int carry = s_inc[63];
    __syncthreads();
    if (tid >= 64 && tid < kMaxGroups) s_inc[tid] += carry;
    __syncthreads();
    total = s_inc[p.G - 1];
    if constexpr (!TILED) {
      // rows outside [offsets[0], offsets[G]) that no group covers are zero
      if (p.zero_uncovered) {
        const int off0 = min(max(p.offsets[0], 0), p.M);
        const int offG = min(max(p.offsets[p.G], off0), p.M);
        const int n = off0 + (p.M - offG);
        for (int i = blockIdx.x; i < n; i += gridDim.x) {
          const int row = i < off0 ? i : offG + (i - off0);
          bool covered = false;
          for (int g = 0; g < p.G; ++g) covered |= row >= s_mb[g] && row < s_me[g];
          if (!covered)
            for (int c = tid; c < p.N; c += kMidThreads) p.C[(int64_t)row * p.ldc + c] = 0;
        }
      }
    }
  }
  // One tile per workgroup, dealt to the XCDs in chunks (gemm_sched.hpp): the grid covers
  // every tile of non-decreasing offsets. Offsets from a caller may overlap and make more
  // tiles, so with row-major weights (those ops) the workgroups go on in grid strides.
  int W = sched_tile_index(blockIdx.x & 7, blockIdx.x >> 3, 0, 1, chunk);
  if constexpr (TILED) {
    if (W < total) mid_tile<TM, TN, SWIGLU, GATHER, TILED>(p, W, NT, s_ring, s_inc, s_mb, s_me);
  } else {
    for (; W < total; W += gridDim.x) {
      mid_tile<TM, TN, SWIGLU, GATHER, TILED>(p, W, NT, s_ring, s_inc, s_mb, s_me);
      __syncthreads();  // the next tile's DMA overwrites the staging
    }
  }
}

template <int TM, int TN, bool SWIGLU, bool GATHER, bool TILED>
static int launch_mid(const GemmArgs& a, hipStream_t st) {
  if (a.M > kMidMaxRows) return fail(DSK_ERR_INVALID_ARG, "mid_gemm: too many rows");
  constexpr int OUT_N = MidCfg<TM, TN, SWIGLU, GATHER, TILED>::OUT_N;
  const int64_t nt = (a.N + OUT_N - 1) / OUT_N;
  const int64_t tiles =
      ((int64_t)(a.M + 32 * TM - 1) / (32 * TM) + (a.offsets != nullptr ? a.G : 0)) * nt;
  if (tiles > INT32_MAX / 2)
    return fail(DSK_ERR_INVALID_ARG, "mid_gemm: too many tiles");
  const int chunk = sched_balanced_chunk((int)tiles, num_cus());
  const int64_t grid = sched_single_workgroups(tiles, chunk);
  hipLaunchKernelGGL((mid_gemm_kernel<TM, TN, SWIGLU, GATHER, TILED>), dim3((unsigned)grid),
                     dim3(kMidThreads), 0, st, a, chunk);
  return check_launch("mid_gemm_kernel");
}

// Whether the 256 x 256 kernels are ahead for groups of about avg rows each (tiled weights,
// no always-on groups among them). A group of just over 128 rows is two tiles here and one
// there, and the time goes in rounds of a tile per CU, one here taking 1 / 1.9 of one there.
// Measured on MI355X, us, here / there:
//   64 experts of 1408, H = 2048, top-6: GEMM1  T = 1200 153 / 174, 1500 191 / 179, 1900
//     201 / 188, 3000 257 / 289, 3500 270 / 295;  GEMM2  T = 1000 78 / 83, 1200 98 / 85,
//     1500 101 / 92, 1900 108 / 99
//   32 of 2048, H = 4096, top-2: GEMM1  T = 2100 263 / 241, 3000 272 / 263;  GEMM2  134 / 115,
//     144 / 129
//   16 of 4096, H = 2048, top-2: GEMM1  T = 1100 136 / 127, 2500 191 / 215, 3300 238 / 227
//   8 of 1408, H = 2048, top-1:  GEMM1  T = 1500 32 / 42, 2500 44 / 41, 3000 53 / 45
//   8 of 14336, H = 4096, top-2: GEMM1  T = 600 424 / 434, 1500 678 / 679, 1700 763 / 726
// From 200 to 256 rows some groups pass 256 and both orders were seen (64 experts top-6,
// T = 2300 205 / 194 and, with other logits, 205 / 233; top-1, T = 14000 211 / 245): left here.
static bool even_groups_want_large(const GemmArgs& a, bool swiglu, int64_t avg) {
  if (avg <= (swiglu ? 128 : 100) || (avg > 200 && avg <= 256)) return false;
  const int64_t cus = num_cus(), nt = (a.N + (swiglu ? 127 : 255)) / (swiglu ? 128 : 256);
  auto rounds = [&](int64_t rows, int64_t bm) {
    return (a.G * nt * ((rows + bm - 1) / bm) + cus - 1) / cus;
  };
  // GEMM2's 512 tiles (64 groups, two on each CU) take a third one from the few groups past
  // 128 rows that 100 rows on average bring
  return 10 * rounds(avg + (swiglu ? 0 : 28), 128) > 19 * rounds(avg, 256);
}

bool mid_gemm_takes(const GemmArgs& a, bool swiglu) {
  const bool gather = a.a_rows != nullptr, grouped = a.offsets != nullptr;
  if (a.N % 32 || a.up_row_offset % 32 || !aligned16(a.C) || a.ldc % 8) return false;
  if (a.a_group_stride || a.c_group_stride || a.C2 != nullptr) return false;
  if (!grouped) return !swiglu && !gather;
  if (gather && !swiglu) return false;
  // Grouped, by average rows per group. Measured on MI355X, us, against the 256 x 256
  // kernels. Tiled weights, in the MoE layer (64 experts top-6 and 2 always-on groups, T
  // tokens, M / G = 0.12 T):
  //   GEMM1  T = 250 138 / 163, 600 159 / 193, 1000 164 / 207, 2000 224 / 231,
  //          3000 316 / 332, 4096 381 / 371, 8192 695 / 677
  //   GEMM2  T = 250 76 / 108, 600 87 / 109, 1000 107 / 114, 1400 117 / 121,
  //          2000 133 / 133, 3000 187 / 185, 4096 221 / 217
  // Row-major weights, the op by op pipeline (64 experts, M / G = 0.094 T):
  //   gate|up  T = 16 124 / 181, 150 156 / 209, 600 164 / 219, 1000 191 / 222, 2000 260 / 239
  //   down     T = 16 50 / 91, 150 67 / 101, 600 80 / 106, 1000 86 / 108, 2000 127 / 119
  const int64_t avg = a.M / (a.G > 0 ? a.G : 1);
  if (a.M > kMidMaxRows) return false;
  if (!a.b_tiled) return avg <= 130;
  // tiled weights come from the fused layer, whose offsets never overlap (the grid holds
  // the tiles of such offsets only)
  return swiglu == gather && a.offsets_sorted && avg <= (swiglu ? 430 : 230) &&
         !(a.even_groups && even_groups_want_large(a, swiglu, avg));
}

int run_mid_gemm(const GemmArgs& a, bool swiglu, hipStream_t st) {
  if (a.offsets == nullptr && a.M > kMidMaxRows) {  // a launch for each kMidMaxRows rows
    for (int r = 0; r < a.M; r += kMidMaxRows) {
      GemmArgs part = a;
      part.M = a.M - r < kMidMaxRows ? a.M - r : kMidMaxRows;
      part.A += (int64_t)r * a.lda;
      part.C += (int64_t)r * a.ldc;
      if (a.rowsq_out != nullptr) part.rowsq_out += r;
      if (a.rowscale_ss != nullptr) part.rowscale_ss += r;
      const int rc = run_mid_gemm(part, swiglu, st);
      if (rc) return rc;
    }
    return DSK_OK;
  }
  const int64_t avg = a.M / (a.offsets != nullptr && a.G > 0 ? a.G : 1);
  const bool gather = a.a_rows != nullptr;
  if (a.offsets != nullptr && !a.b_tiled) {
    // 64-row tiles while most groups fit one (T = 600: gate|up 164 us against 183 with 128)
    if (avg <= 70) {
      if (swiglu) return gather ? launch_mid<2, 1, true, true, false>(a, st)
                                : launch_mid<2, 1, true, false, false>(a, st);
      return launch_mid<2, 1, false, false, false>(a, st);
    }
    if (swiglu) return gather ? launch_mid<4, 1, true, true, false>(a, st)
                              : launch_mid<4, 1, true, false, false>(a, st);
    return launch_mid<4, 1, false, false, false>(a, st);
  }
  if (swiglu) return launch_mid<4, 2, true, true, true>(a, st);
  if (a.offsets != nullptr) {
    // few rows per group: 64-row tiles, and half the weight rows per workgroup, which
    // spreads the weight stream over twice the workgroups (T = 250: 76 us against 91). Even
    // groups of more than 50 rows begin to pass 64, and stay whole where one 128-row tile
    // each is at most two per CU but covers them (64 experts top-6, no always-on groups:
    // T = 600 81 us with 64 rows, 73 with 128; 700 94, 74; 800 96, 75).
    const int64_t wide = a.G * (int64_t)((a.N + 255) / 256), ncu = num_cus();
    const bool whole = a.even_groups && avg > 50 && wide >= ncu && wide <= 2 * ncu;
    if (avg <= 80 && !whole) return launch_mid<2, 1, false, false, true>(a, st);
    return launch_mid<4, 2, false, false, true>(a, st);
  }
  // Dense: the tile with the least estimated time, from c = tiles on the fullest CU.
  // The coefficients follow the times at K = 2048 (token rows x weight rows; tiled:
  // 64 x 128 13 us a tile, 64 x 256 17.5, 128 x 256 27; row-major: 64 x 128 2 + 10.5 c,
  // 128 x 128 9 + 15 c); over M = 65..8192 and the layer's three (N, K) the choice was
  // the fastest tile or within 12 % of it. Measured against the 256 x 256 kernels:
  // tiled N = 2048, K = 2048: M = 257 15 / 282 us, 1111 19 / 166, 4096 36 / 54, 8192
  // 61 / 70; N = 3648: M = 1111 30 / 89, 4096 62 / 101, 16384 228 / 242; N = 4096, K = 512:
  // M = 1111 12.5 / 34, 16384 81 / 87. Row-major N = 3648: M = 257 14 / 128, 1111 31 / 81,
  // 8192 129 / 202.
  const int64_t cus = num_cus();
  auto tiles_per_cu = [&](int bm, int bn) {
    const int64_t t = (int64_t)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
    return (double)((t + cus - 1) / cus);
  };
  if (!a.b_tiled)
    return 2.0 + 10.5 * tiles_per_cu(64, 128) <= 9.0 + 15.0 * tiles_per_cu(128, 128)
               ? launch_mid<2, 1, false, false, false>(a, st)
               : launch_mid<4, 1, false, false, false>(a, st);
  const bool row_stats = a.rowsq_out != nullptr || a.rowscale_ss != nullptr;  // whole 256 columns
  const double c64w = 17.5 * tiles_per_cu(64, 256), c128w = 27.0 * tiles_per_cu(128, 256);
  if (!row_stats && 13.0 * tiles_per_cu(64, 128) < (c64w < c128w ? c64w : c128w))
    return launch_mid<2, 1, false, false, true>(a, st);
  return c64w < c128w ? launch_mid<2, 2, false, false, true>(a, st)
                      : launch_mid<4, 2, false, false, true>(a, st);
}

}  // namespace dsk
