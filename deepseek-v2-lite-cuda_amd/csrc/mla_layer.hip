// The MLA module as one C call each for its two hot forms, on DeepSeek-V2-Lite's
// dims (heads of 128 + 64 / 128, latent 512) and fragment-tiled weights: the full
// sequence (DeepSeekMLA.forward, src/reference/mla.py:295-393) and a decode step of
// up to 64 new tokens against the latent cache. They only enqueue the kernels of the
// other files on the caller's stream, with every intermediate in one workspace: a
// decode step is 6 launches of 3-8 us each, and issuing them one Python op at a time
// took ~110 us per step, four times their GPU time.
#include "dsk_internal.hpp"

namespace dsk {

constexpr int kMlaNope = 128, kMlaRope = 64, kMlaV = 128, kMlaLora = 512;
constexpr int kMlaHeads = 16;     // of the decode attention
constexpr int kRowsTokens = 4;    // decode steps up to this many tokens: vector-ALU row kernel
constexpr int kDecodeTokens = 64; // largest native decode step

struct Carver {
  size_t off = 0;
  size_t take(size_t bytes) {
    const size_t o = off;
    off += align_up(bytes > 0 ? bytes : 1, 256);
    return o;
  }
};

struct ForwardLayout {
  size_t y, ss, kv, k_rot, o, total;
};
static ForwardLayout forward_layout(int64_t rows, int heads) {
  ForwardLayout l{};
  Carver c;
  l.y = c.take((size_t)rows * (heads * (kMlaNope + kMlaRope) + kMlaLora + kMlaRope) * 2);
  l.ss = c.take((size_t)rows * (kMlaLora / 256) * 4);
  l.kv = c.take((size_t)rows * heads * (kMlaNope + kMlaV) * 2);
  l.k_rot = c.take((size_t)rows * kMlaRope * 2);
  l.o = c.take((size_t)rows * heads * kMlaV * 2);
  l.total = c.off;
  return l;
}

struct DecodeLayout {
  size_t q, q_abs, o_lat, o, attn, total;
};
static DecodeLayout decode_layout(int batch, int n, int kv_len) {
  DecodeLayout l{};
  Carver c;
  const size_t T = (size_t)batch * n;
  l.q = c.take(T * kMlaHeads * (kMlaNope + kMlaRope) * 2);
  l.q_abs = c.take(T * kMlaHeads * kMlaLora * 2);
  l.o_lat = c.take(T * kMlaHeads * kMlaLora * 2);
  l.o = c.take(T * kMlaHeads * kMlaV * 2);
  l.attn = c.take(dsk_mla_decode_workspace_size(batch, n, kv_len));
  l.total = c.off;
  return l;
}

}  // namespace dsk

using namespace dsk;

extern "C" size_t dsk_mla_forward_workspace_size(int batch, int seq, int heads) {
  if (batch <= 0 || seq <= 0 || heads <= 0) return 256;
  return forward_layout((int64_t)batch * seq, heads).total;
}

extern "C" int dsk_mla_forward(const dsk_bf16* x, const dsk_bf16* w_q_kva, const dsk_bf16* w_kvb,
                               const dsk_bf16* w_o, const dsk_bf16* cos_t, const dsk_bf16* sin_t,
                               int64_t ld_cs, int64_t cs_batch_stride, float eps, float scale,
                               int causal, const void* mask, int mask_dtype, int64_t mask_sb,
                               int64_t mask_sh, int64_t mask_sq, dsk_bf16* out, int batch,
                               int seq, int heads, int hidden, void* workspace, size_t bytes,
                               void* stream) {
  DSK_REQUIRE(batch >= 0 && seq >= 0 && heads > 0 && hidden > 0, DSK_ERR_INVALID_ARG,
              "mla_forward: invalid sizes");
  DSK_REQUIRE(heads % 4 == 0, DSK_ERR_INVALID_ARG, "mla_forward: heads must be a multiple of 4");
  DSK_REQUIRE((int64_t)batch * seq < (int64_t)INT32_MAX, DSK_ERR_INVALID_ARG,
              "mla_forward: too many tokens");
  const int rows = batch * seq;
  if (rows == 0) return DSK_OK;
  const ForwardLayout l = forward_layout(rows, heads);
  DSK_REQUIRE(workspace != nullptr && aligned16(workspace) && bytes >= l.total, DSK_ERR_WORKSPACE,
              "mla_forward: workspace too small");
  char* ws = static_cast<char*>(workspace);
  dsk_bf16* y = reinterpret_cast<dsk_bf16*>(ws + l.y);
  float* ss = reinterpret_cast<float*>(ws + l.ss);
  dsk_bf16* kv = reinterpret_cast<dsk_bf16*>(ws + l.kv);
  dsk_bf16* k_rot = reinterpret_cast<dsk_bf16*>(ws + l.k_rot);
  dsk_bf16* o = reinterpret_cast<dsk_bf16*>(ws + l.o);
  const int nq = heads * (kMlaNope + kMlaRope), ny = nq + kMlaLora + kMlaRope;
  const int nkv = heads * (kMlaNope + kMlaV), no = heads * kMlaV;
  const dsk_bf16* k_pe = y + nq + kMlaLora;
  int rc = dsk_linear_rowsq(x, hidden, w_q_kva, y, ny, rows, hidden, ny, ss, rows, nq,
                            nq + kMlaLora, stream);
  if (rc) return rc;
  rc = dsk_linear_rowscale(y + nq, ny, w_kvb, kv, nkv, rows, kMlaLora, nkv, ss, rows,
                           kMlaLora / 256, kMlaLora, eps, stream);
  if (rc) return rc;
  rc = dsk_rope(k_pe, (int64_t)seq * ny, 0, ny, cos_t, sin_t, cs_batch_stride, ld_cs, k_rot,
                batch, 1, seq, kMlaRope, stream);
  if (rc) return rc;
  rc = dsk_mla_prefill_attention(y, ny, kv, nkv, k_rot, kMlaRope, (int64_t)seq * kMlaRope, cos_t,
                                 sin_t, ld_cs, cs_batch_stride, scale, causal, mask, mask_dtype,
                                 mask_sb, mask_sh, mask_sq, o, no, batch, seq, seq, heads, stream);
  if (rc) return rc;
  return dsk_linear_ex(o, no, w_o, DSK_LAYOUT_TILED, out, hidden, rows, no, hidden, stream);
}

extern "C" size_t dsk_mla_decode_forward_workspace_size(int batch, int n, int kv_len) {
  if (batch <= 0 || n <= 0 || kv_len <= 0) return 256;
  return decode_layout(batch, n, kv_len).total;
}

extern "C" int dsk_mla_decode_forward(const dsk_bf16* x, const dsk_bf16* w_q_kva,
                                      const dsk_bf16* w_uk, const dsk_bf16* w_uv,
                                      const dsk_bf16* w_o, dsk_bf16* cache_rows, int64_t ld_tok,
                                      int64_t ld_batch, const dsk_bf16* cos_t,
                                      const dsk_bf16* sin_t, float eps, float scale, int batch,
                                      int n, int cached, int rope_len, int hidden, dsk_bf16* out,
                                      void* workspace, size_t bytes, void* stream) {
  DSK_REQUIRE(batch >= 0 && n >= 0 && cached >= 0 && hidden > 0, DSK_ERR_INVALID_ARG,
              "mla_decode_forward: invalid sizes");
  if (batch == 0 || n == 0) return DSK_OK;
  DSK_REQUIRE((batch == 1 || n == 1) && (int64_t)batch * n <= kDecodeTokens, DSK_ERR_INVALID_ARG,
              "mla_decode_forward: one sequence or one token each, at most 64 tokens");
  DSK_REQUIRE(cache_rows != nullptr && ld_tok >= kMlaLora + 2 * kMlaRope, DSK_ERR_INVALID_ARG,
              "mla_decode_forward: cache rows must hold 640 values");
  const int L = cached + n, T = batch * n;
  const DecodeLayout l = decode_layout(batch, n, L);
  DSK_REQUIRE(workspace != nullptr && aligned16(workspace) && bytes >= l.total, DSK_ERR_WORKSPACE,
              "mla_decode_forward: workspace too small");
  char* ws = static_cast<char*>(workspace);
  dsk_bf16* q = reinterpret_cast<dsk_bf16*>(ws + l.q);
  dsk_bf16* q_abs = reinterpret_cast<dsk_bf16*>(ws + l.q_abs);
  dsk_bf16* o_lat = reinterpret_cast<dsk_bf16*>(ws + l.o_lat);
  dsk_bf16* o = reinterpret_cast<dsk_bf16*>(ws + l.o);
  constexpr int hd = kMlaNope + kMlaRope, nq = kMlaHeads * hd, nkva = kMlaLora + kMlaRope;
  constexpr int no = kMlaHeads * kMlaV;
  // kv_a's output goes straight into the cache slots of the new tokens
  dsk_bf16* slots = cache_rows + (int64_t)cached * ld_tok;
  const int64_t slot_stride = batch == 1 ? ld_tok : ld_batch;
  const bool few = T <= kRowsTokens;
  int rc = few ? dsk_linear_rows(x, hidden, 0, w_q_kva, 0, q, nq, 0, slots, slot_stride, 0, nq, 1,
                                 T, hidden, nq + nkva, stream)
               : dsk_linear_split(x, hidden, w_q_kva, q, nq, slots, slot_stride, T, hidden,
                                  nq + nkva, nq, stream);
  if (rc) return rc;
  // per head: q_abs[h] = (W_UK[h] w)^T q_nope[h], into [head][token][512]
  rc = few ? dsk_linear_rows(q, nq, hd, w_uk, (int64_t)kMlaLora * kMlaNope, q_abs, kMlaLora,
                             (int64_t)T * kMlaLora, nullptr, 0, 0, kMlaLora, kMlaHeads, T,
                             kMlaNope, kMlaLora, stream)
           : dsk_linear_batched(q, nq, hd, w_uk, q_abs, kMlaLora, (int64_t)T * kMlaLora, kMlaHeads,
                                T, kMlaNope, kMlaLora, stream);
  if (rc) return rc;
  rc = dsk_mla_decode_attention(q_abs, kMlaLora, (int64_t)T * kMlaLora, q + kMlaNope, nq, hd,
                                cache_rows, cache_rows + kMlaLora, cache_rows + nkva, rope_len,
                                ld_tok, batch > 1 ? ld_batch : (int64_t)L * ld_tok, cos_t, sin_t,
                                eps, scale, batch, n, L, o_lat, kMlaLora, (int64_t)T * kMlaLora,
                                ws + l.attn, bytes - l.attn, stream);
  if (rc) return rc;
  // o[t, 128 h ..] = (W_UV[h] w) o_lat[h, t], token-major
  rc = few ? dsk_linear_rows(o_lat, kMlaLora, (int64_t)T * kMlaLora, w_uv,
                             (int64_t)kMlaV * kMlaLora, o, no, kMlaV, nullptr, 0, 0, kMlaV,
                             kMlaHeads, T, kMlaLora, kMlaV, stream)
           : dsk_linear_batched(o_lat, kMlaLora, (int64_t)T * kMlaLora, w_uv, o, no, kMlaV,
                                kMlaHeads, T, kMlaLora, kMlaV, stream);
  if (rc) return rc;
  return few ? dsk_linear_rows(o, no, 0, w_o, 0, out, hidden, 0, nullptr, 0, 0, hidden, 1, T, no,
                               hidden, stream)
             : dsk_linear_ex(o, no, w_o, DSK_LAYOUT_TILED, out, hidden, T, no, hidden, stream);
}
