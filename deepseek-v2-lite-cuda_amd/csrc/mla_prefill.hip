// Fused causal / masked MLA attention over up-projected K and V (gfx950): the
// attention of DeepSeekMLA.forward (src/reference/mla.py:354-384) for the last
// n of L positions, straight from the projection rows.
//
//   score(i, j) = scale * (q_nope_i . k_nope_j + rope_i(q_pe_i) . k_rope_j) (+ mask)
//   out(i)      = sum_j softmax_j(score(i, .)) v_j
//
// q rows are the q projection's (per head 128 nope | 64 raw RoPE values, rotated
// here), kv rows the kv_b projection's (per head 128 k_nope | 128 v) and k_rope
// the rotated shared keys. Scores, the running max and sum and the output stay
// in fp32 registers; only the probabilities are rounded to bf16 for P.V, so no
// score is ever stored.
//
// One workgroup owns 32 NW query rows of one head, 32 per wave, and walks the
// keys in tiles of 64. A tile (k_nope 16 KB, v 16 KB, k_rope 8 KB) lands in one
// of two LDS buffers by global->LDS DMA while the previous one is used, and one
// barrier per tile publishes it and frees the other. Both products run
// transposed on v_mfma_f32_32x32x16_bf16:
//   S^T[key][query] = K Q^T: K rows are 16-byte LDS reads in operand order, the
//     wave's 32 queries stay in registers (48). A lane then holds 32 of the 64
//     scores of ONE query, so max, sum and rescale are in-lane work plus one swap
//     with lane + 32.
//   O^T[dim][query] += V^T P^T: the score layout is the operand layout of P^T up
//     to an order of the keys inside a step of 16 (slot 8h + j is key 8 (j / 4) +
//     4h + j % 4), and V^T is read in that order by the transposing LDS read
//     (ds_read_b64_tr_b16: 4 keys x 16 dims per 16 lanes), so P never moves
//     between lanes.
// LDS rows are swizzled in 16-byte chunks (the DMA lane fetches the chunk its
// slot stands for): K rows by key % 16, RoPE rows as the GEMM's 128-byte rows, V
// rows by 4 (key % 4), which keeps the 4-row transposing reads on distinct banks.
//
// Bound: the two products (320 multiply-adds per score) on the matrix cores,
// with ~30 VALU cycles per wave-wide score register beside them; two waves per
// SIMD overlap the one wave's softmax with the other's MFMAs. Measured on MI355X
// against the torch products around a softmax pass that this replaces (both
// products, softmax and operand packing): b = 4, s = 2048, 16 heads, causal 672 ->
// 137 us (653 TFLOP/s of the causal half); b = 2, s = 1111 169 -> 44 us (the RoPE
// launch of k_pe included in both new figures).
#include "dsk_common.hpp"

#include <math.h>

#include <algorithm>
#include <cstring>

namespace dsk {

constexpr int kPfNope = 128, kPfRope = 64, kPfV = 128;
constexpr int kPfQ = kPfNope + kPfRope;  // one head's slice of a q row
constexpr int kPfKV = kPfNope + kPfV;    // one head's slice of a kv row
constexpr int kPfTile = 64;              // keys per tile
constexpr int kPfRopeOff = kPfTile * kPfNope * 2;             // 16 KB of k_nope first
constexpr int kPfVOff = kPfRopeOff + kPfTile * kPfRope * 2;   // then 8 KB of k_rope
constexpr int kPfBuf = kPfVOff + kPfTile * kPfV * 2;          // then 16 KB of v: 40 KB

struct PrefillArgs {
  const uint16_t* q;      // query row t (batch-major) at t * ld_q
  int64_t ld_q;
  const uint16_t* kv;     // key row at (b * L + j) * ld_kv
  int64_t ld_kv;
  const uint16_t* krope;  // rotated key at b * kr_bs + j * ld_kr
  int64_t ld_kr, kr_bs;
  const uint16_t* cos_t;  // row = position, b * cs_bs + pos * ld_cs
  const uint16_t* sin_t;
  int64_t ld_cs, cs_bs;
  uint16_t* out;          // row t, head h at t * ld_out + h * 128
  int64_t ld_out;
  int n, L, heads, causal;
  float scale;
  const void* mask;       // additive, (b, h, query) strides, key stride 1
  int64_t mask_sb, mask_sh, mask_sq;
};

typedef short s16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8_t lds_frag(uint32_t byte_addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>(
      (uintptr_t)byte_addr);
}
// 4 keys of one dim from 4 rows of 16 dims (the 16 lanes of a row supply them)
__device__ __forceinline__ s16x4_t lds_read_tr(uint32_t byte_addr) {
  typedef __attribute__((address_space(3))) s16x4_t lds_t;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t*)(uintptr_t)byte_addr);
}
// max / sum over lanes l and l ^ 32, on both
__device__ __forceinline__ float pair_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Four consecutive mask elements as floats; keys from kv_len on are not read.
template <typename T>
__device__ __forceinline__ void load_mask4(const T* p, int key, int kv_len, float (&m)[4]) {
  T raw[4];
  if (key + 4 <= kv_len) {
    __builtin_memcpy(raw, p + key, sizeof raw);  // rows need not be aligned
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c) raw[c] = key + c < kv_len ? p[key + c] : T(0);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if constexpr (sizeof(T) == 2) m[c] = bf16_to_f32(raw[c]);
    else m[c] = raw[c];
  }
}

// MASK: 0 none, 1 bf16, 2 fp32.
template <int NW, int MASK>
__global__ __launch_bounds__(64 * NW, 2) void prefill_attn_kernel(PrefillArgs a) {
  __shared__ __attribute__((aligned(1024))) char s_buf[2 * kPfBuf];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h32 = lane >> 5, r32 = lane & 31;
  const int b = blockIdx.x / a.heads, head = blockIdx.x - b * a.heads;
  // the longest (last) query blocks first, so the short ones fill the tail
  const int q0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * 32 * NW;
  const int off = a.L - a.n;  // position of query 0
  const int wq0 = q0 + 32 * wave;
  const int qi = wq0 + r32;                 // this lane's query
  const int qc = min(qi, a.n - 1);
  const int last_key = a.causal ? min(qi + off, a.L - 1) : a.L - 1;  // last visible key
  const int k_end = a.causal ? min(a.L, q0 + 32 * NW + off) : a.L;   // of the workgroup
  const int ntiles = (k_end + kPfTile - 1) / kPfTile;
  // tiles of this wave: [0, w_tiles), those from w_full on need the key limit
  const int w_end = a.causal ? min(a.L, wq0 + 32 + off) : a.L;
  const int w_tiles = wq0 < a.n ? (w_end + kPfTile - 1) / kPfTile : 0;
  const int w_full = (a.causal ? min(a.L, wq0 + off + 1) : a.L) / kPfTile;

  // ---- tile DMA: 40 instructions of 1 KB (16 k_nope, 16 v, 8 rope), NW apart
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(s_buf));
  const char* kv_b = reinterpret_cast<const char*>(
      a.kv + (int64_t)b * a.L * a.ld_kv + head * kPfKV);
  const char* kr_b = reinterpret_cast<const char*>(a.krope + b * a.kr_bs);
  const uint32_t ldkv2 = (uint32_t)a.ld_kv * 2, ldkr2 = (uint32_t)a.ld_kr * 2;
  const int row4 = lane >> 4, row8 = lane >> 3;
  const uint32_t c_k = (uint32_t)((lane & 15) ^ ((4 * wave + row4) & 15)) * 16;
  const uint32_t c_v = (uint32_t)((lane & 15) ^ (row4 << 2)) * 16 + kPfNope * 2;
  const uint32_t c_r = (uint32_t)((lane & 7) ^ row8 ^ (wave & 1)) * 16;
  // Eight waves: a running 64-bit base and fixed 32-bit offsets inside the tile (the last
  // tile's rows past the end are clamped), so that a sequence may span any size. Four waves,
  // one per SIMD, have nothing to cover the scalar steps and the branch with, and the address
  // arithmetic between two DMA instructions is free there (s = 2000 53.8 -> 56.1 us without
  // it, where eight waves gain, s = 4096 143.0 -> 140.8): they address all of a sequence of
  // less than 4 GiB from its start.
  constexpr bool kRunning = NW == 8;
  uint32_t off_k[16 / NW], off_v[16 / NW], off_r[8 / NW];
  auto tile_offsets = [&](int last) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 16 / NW; ++j) {
      const uint32_t row = (uint32_t)min(4 * (wave + NW * j) + row4, last) * ldkv2;
      off_k[j] = row + c_k;
      off_v[j] = row + c_v;
    }
#pragma unroll
    for (int j = 0; j < 8 / NW; ++j)
      off_r[j] = (uint32_t)min(8 * (wave + NW * j) + row8, last) * ldkr2 + c_r;
  };
  if constexpr (kRunning) tile_offsets(min(kPfTile, a.L) - 1);
  const int whole = a.L / kPfTile;  // tiles without rows past the end
  const char *kv_t = kv_b, *kr_t = kr_b;
  auto dma_tile = [&](int t, uint32_t buf) __attribute__((always_inline)) {
    const int k0 = t * kPfTile;
    if constexpr (kRunning) {
      if (t == whole) tile_offsets(a.L - 1 - k0);  // uniform, at most once
    }
#pragma unroll
    for (int j = 0; j < 16 / NW; ++j) {
      const int i = wave + NW * j;
      if constexpr (kRunning) {
        dma_1kb(kv_t, off_k[j], buf + i * 1024);
        dma_1kb(kv_t, off_v[j], buf + kPfVOff + i * 1024);
      } else {
        const uint32_t row = (uint32_t)min(k0 + 4 * i + row4, a.L - 1) * ldkv2;
        dma_1kb(kv_b, row + c_k, buf + i * 1024);
        dma_1kb(kv_b, row + c_v, buf + kPfVOff + i * 1024);
      }
    }
#pragma unroll
    for (int j = 0; j < 8 / NW; ++j) {
      const int i = wave + NW * j;
      if constexpr (kRunning)
        dma_1kb(kr_t, off_r[j], buf + kPfRopeOff + i * 1024);
      else
        dma_1kb(kr_b, (uint32_t)min(k0 + 8 * i + row8, a.L - 1) * ldkr2 + c_r,
                buf + kPfRopeOff + i * 1024);
    }
    if constexpr (kRunning) {
      kv_t += (int64_t)kPfTile * ldkv2;
      kr_t += (int64_t)kPfTile * ldkr2;
    }
  };
  dma_tile(0, lds0);

  // ---- query fragments: step s holds dims 16 s + 8 h32 .. + 7 of query r32
  bf16x8_t qf[kPfQ / 16];
  {
    const uint16_t* qr = a.q + ((int64_t)b * a.n + qc) * a.ld_q + head * kPfQ;
#pragma unroll
    for (int s = 0; s < kPfNope / 16; ++s)
      qf[s] = *reinterpret_cast<const bf16x8_t*>(qr + 16 * s + 8 * h32);
    const int64_t trow = b * a.cs_bs + (int64_t)(off + qc) * a.ld_cs;
#pragma unroll
    for (int u = 0; u < 2; ++u) {  // rotated pieces c and 4 + c of c = h32, 2 + h32
      const int c = 2 * u + h32;
      const u32x4_t x[2] = {*reinterpret_cast<const u32x4_t*>(qr + kPfNope + 16 * c),
                            *reinterpret_cast<const u32x4_t*>(qr + kPfNope + 16 * c + 8)};
      const uint16_t* ct = a.cos_t + trow + 8 * c;
      const uint16_t* st = a.sin_t + trow + 8 * c;
      u32x4_t lo, hi;
      rope_pieces(x, *reinterpret_cast<const u32x4_t*>(ct),
                  *reinterpret_cast<const u32x4_t*>(ct + kPfRope / 2),
                  *reinterpret_cast<const u32x4_t*>(st),
                  *reinterpret_cast<const u32x4_t*>(st + kPfRope / 2), lo, hi);
      qf[8 + u] = __builtin_bit_cast(bf16x8_t, lo);
      qf[10 + u] = __builtin_bit_cast(bf16x8_t, hi);
    }
  }

  constexpr float kLog2e = 1.44269504088896340736f;
  const float c_exp = MASK ? kLog2e : a.scale * kLog2e;  // exponent of 2 per unit of score
  const int64_t mrow = MASK ? b * a.mask_sb + head * a.mask_sh + qc * a.mask_sq : 0;

  floatx16_t o[4];  // dims 32 db + 8 (i / 4) + 4 h32 + i % 4 of query r32
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's share

  // LDS read addresses inside a buffer
  const uint32_t ka = (uint32_t)r32 * 256;                     // + 32 kb rows
  const uint32_t ra = (uint32_t)kPfRopeOff + r32 * 128;
  const int kx = r32 & 15, rx = (r32 & 7) ^ ((r32 >> 3) & 1);
  const int l16 = lane & 15, vr = l16 >> 2;
  const uint32_t va = (uint32_t)kPfVOff + (4 * h32 + vr) * 256 +
                      (2 * ((lane >> 4) & 1) + ((l16 >> 1) & 1)) * 16 + (l16 & 1) * 8;

#pragma unroll 1
  for (int t = 0; t < ntiles; ++t) {
    const uint32_t buf = lds0 + (t & 1) * kPfBuf;
    // tile t has landed (every wave waits for its own DMA), and every wave is
    // past its reads of tile t - 1, whose buffer tile t + 1 now fills
    wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + 1 < ntiles) dma_tile(t + 1, lds0 + ((t + 1) & 1) * kPfBuf);
    if (t >= w_tiles) continue;  // uniform over the wave

    floatx16_t s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < kPfQ / 16; ++ks) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const uint32_t ad =
            ks < 8 ? buf + ka + kb * 32 * 256 + (uint32_t)((2 * ks + h32) ^ kx) * 16
                   : buf + ra + kb * 32 * 128 + (uint32_t)((2 * (ks - 8) + h32) ^ rx) * 16;
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_frag(ad), qf[ks], s[kb], 0, 0, 0);
      }
    }

    // ---- mask and online softmax; score (kb, i) is key k0 + 32 kb + 8 (i / 4) + i % 4
    const int k0 = t * kPfTile + 4 * h32;
    if constexpr (MASK != 0) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float mv[4];
          if constexpr (MASK == 1)
            load_mask4(reinterpret_cast<const uint16_t*>(a.mask) + mrow, k0 + 32 * kb + 8 * g, a.L, mv);
          else
            load_mask4(reinterpret_cast<const float*>(a.mask) + mrow, k0 + 32 * kb + 8 * g, a.L, mv);
#pragma unroll
          for (int c = 0; c < 4; ++c) s[kb][4 * g + c] = s[kb][4 * g + c] * a.scale + mv[c];
        }
    }
    if (t >= w_full) {  // uniform
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (k0 + 32 * kb + 8 * (i >> 2) + (i & 3) > last_key) s[kb][i] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
    const float m_new = fmaxf(m_run, pair_max(mx));
    const float m_ref = m_new == -INFINITY ? 0.f : m_new;  // nothing visible yet
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_ref) * c_exp);
    m_run = m_new;
    const float m_c = m_ref * c_exp;
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        // with a mask the difference comes first: mask values near the type's
        // lowest overflow when scaled
        s[kb][i] = __builtin_amdgcn_exp2f(MASK ? (s[kb][i] - m_ref) * c_exp
                                               : fmaf(s[kb][i], c_exp, -m_c));
        sum += s[kb][i];
      }
    l_run = fmaf(l_run, alpha, sum);
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }

    // ---- O^T += V^T P^T, 16 keys a step
#pragma unroll
    for (int kg = 0; kg < 4; ++kg) {
      u32x4_t pw;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        pw[c] = pack_bf16x2(s[kg >> 1][8 * (kg & 1) + 2 * c], s[kg >> 1][8 * (kg & 1) + 2 * c + 1]);
      const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, pw);
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const uint32_t ad = buf + va + (uint32_t)(db ^ vr) * 64 + kg * 16 * 256;
        const s16x4_t lo = lds_read_tr(ad), hi = lds_read_tr(ad + 8 * 256);
        typedef short s16x8_t __attribute__((ext_vector_type(8)));
        const s16x8_t vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vf), pf,
                                                        o[db], 0, 0, 0);
      }
    }
  }

  // ---- epilogue: one swap of lane halves per pair of 4-dim groups gives each
  // lane 8 consecutive dims (16-byte stores). A row with no visible key has sum
  // 0 and comes out NaN, as softmax over all -inf does.
  const float inv = 1.f / pair_sum(l_run);
  if (qi >= a.n) return;  // the same for lanes l and l + 32
  uint16_t* orow = a.out + ((int64_t)b * a.n + qi) * a.ld_out + head * kPfV;
#pragma unroll
  for (int db = 0; db < 4; ++db) {
#pragma unroll
    for (int q2 = 0; q2 < 2; ++q2) {
      uint32_t w[2][2];
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          w[g][c] = pack_bf16x2(o[db][8 * q2 + 4 * g + 2 * c] * inv,
                                o[db][8 * q2 + 4 * g + 2 * c + 1] * inv);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const auto r = __builtin_amdgcn_permlane32_swap(w[0][c], w[1][c], false, false);
        w[0][c] = r[0];
        w[1][c] = r[1];
      }
      *reinterpret_cast<u32x4_t*>(orow + 32 * db + 16 * q2 + 8 * h32) =
          u32x4_t{w[0][0], w[0][1], w[1][0], w[1][1]};
    }
  }
}

template <int NW>
static void launch_prefill(const PrefillArgs& a, int batch, int mask_kind, hipStream_t st) {
  const dim3 grid((unsigned)(batch * a.heads), (unsigned)((a.n + 32 * NW - 1) / (32 * NW)));
  if (mask_kind == 0)
    hipLaunchKernelGGL((prefill_attn_kernel<NW, 0>), grid, dim3(64 * NW), 0, st, a);
  else if (mask_kind == 1)
    hipLaunchKernelGGL((prefill_attn_kernel<NW, 1>), grid, dim3(64 * NW), 0, st, a);
  else
    hipLaunchKernelGGL((prefill_attn_kernel<NW, 2>), grid, dim3(64 * NW), 0, st, a);
}

}  // namespace dsk

using namespace dsk;

extern "C" int dsk_mla_prefill_attention(
    const dsk_bf16* q, int64_t ld_q, const dsk_bf16* kv, int64_t ld_kv, const dsk_bf16* k_rope,
    int64_t ld_kr, int64_t kr_batch_stride, const dsk_bf16* cos_t, const dsk_bf16* sin_t,
    int64_t ld_cs, int64_t cs_batch_stride, float scale, int causal, const void* mask,
    int mask_dtype, int64_t mask_sb, int64_t mask_sh, int64_t mask_sq, dsk_bf16* out,
    int64_t ld_out, int batch, int q_len, int kv_len, int heads, void* stream) {
  DSK_REQUIRE(batch >= 0 && q_len >= 0 && heads >= 0, DSK_ERR_INVALID_ARG,
              "mla_prefill_attention: negative size");
  if (batch == 0 || q_len == 0 || heads == 0) return DSK_OK;
  DSK_REQUIRE(kv_len >= q_len, DSK_ERR_INVALID_ARG,
              "mla_prefill_attention: need q_len <= kv_len (the queries are the last positions)");
  DSK_REQUIRE(q && kv && k_rope && cos_t && sin_t && out, DSK_ERR_NULL_PTR,
              "mla_prefill_attention: NULL pointer");
  DSK_REQUIRE(scale > 0.f, DSK_ERR_INVALID_ARG, "mla_prefill_attention: scale must be positive");
  DSK_REQUIRE(mask == nullptr || mask_dtype == DSK_DTYPE_BF16 || mask_dtype == DSK_DTYPE_F32,
              DSK_ERR_INVALID_ARG,
              "mla_prefill_attention: mask dtype must be DSK_DTYPE_BF16 or DSK_DTYPE_F32");
  DSK_REQUIRE(aligned16(q) && aligned16(kv) && aligned16(k_rope) && aligned16(cos_t) &&
                  aligned16(sin_t) && aligned16(out) && ld_q % 8 == 0 && ld_kv % 8 == 0 &&
                  ld_kr % 8 == 0 && kr_batch_stride % 8 == 0 && ld_cs % 8 == 0 &&
                  cs_batch_stride % 8 == 0 && ld_out % 8 == 0,
              DSK_ERR_ALIGNMENT, "mla_prefill_attention: rows must be 16-byte aligned");
  DSK_REQUIRE(ld_q >= (int64_t)heads * kPfQ && ld_kv >= (int64_t)heads * kPfKV &&
                  ld_kr >= kPfRope && ld_cs >= kPfRope && ld_out >= (int64_t)heads * kPfV &&
                  kr_batch_stride >= 0 && cs_batch_stride >= 0,
              DSK_ERR_INVALID_ARG, "mla_prefill_attention: row stride smaller than the row");
  // the rows of one tile are addressed by 32-bit byte offsets
  const int64_t tile_rows = std::min(kv_len, kPfTile);
  DSK_REQUIRE(tile_rows * ld_kv * 2 < ((int64_t)1 << 32) && tile_rows * ld_kr * 2 < ((int64_t)1 << 32),
              DSK_ERR_INVALID_ARG, "mla_prefill_attention: 64 key rows must span less than 4 GiB");
  DSK_REQUIRE((int64_t)batch * heads <= INT32_MAX && q_len <= 65535 * 128, DSK_ERR_INVALID_ARG,
              "mla_prefill_attention: too many query blocks");
  PrefillArgs a;
  a.q = reinterpret_cast<const uint16_t*>(q);
  a.ld_q = ld_q;
  a.kv = reinterpret_cast<const uint16_t*>(kv);
  a.ld_kv = ld_kv;
  a.krope = reinterpret_cast<const uint16_t*>(k_rope);
  a.ld_kr = ld_kr;
  a.kr_bs = kr_batch_stride;
  a.cos_t = reinterpret_cast<const uint16_t*>(cos_t);
  a.sin_t = reinterpret_cast<const uint16_t*>(sin_t);
  a.ld_cs = ld_cs;
  a.cs_bs = cs_batch_stride;
  a.out = reinterpret_cast<uint16_t*>(out);
  a.ld_out = ld_out;
  a.n = q_len;
  a.L = kv_len;
  a.heads = heads;
  a.causal = causal != 0;
  a.scale = scale;
  a.mask = mask;
  a.mask_sb = mask_sb;
  a.mask_sh = mask_sh;
  a.mask_sq = mask_sq;
  const int mask_kind = mask == nullptr ? 0 : mask_dtype == DSK_DTYPE_BF16 ? 1 : 2;
  // 256-query workgroups read each K/V tile from the L2 half as often; below one
  // per CU, 128-query ones (two per CU) spread the work further, if 32-bit offsets
  // reach the whole sequence
  const int64_t wide = (int64_t)batch * heads * ((q_len + 255) / 256);
  const bool far = (int64_t)kv_len * std::max(ld_kv, ld_kr) * 2 >= ((int64_t)1 << 32);
  if (wide >= 256 || far)
    launch_prefill<8>(a, batch, mask_kind, as_stream(stream));
  else
    launch_prefill<4>(a, batch, mask_kind, as_stream(stream));
  return check_launch("prefill_attn_kernel");
}
