// A whole pre-norm layer of the 32-bit path in one call: RMSNorm, q/k/v product, q/k norm with rotation and cache write, attention,
// output product, RMSNorm, gate and up product, activation, down product: the launches that their own entry points make, one
// after another on one stream.  What bounds a step of few tokens is the host: asked for one by one from Python, with a tensor made and
// checked for each, a launch takes the host 12 us, from here 2 to 3.
#include <algorithm>
#include "common.h"

SYN_EXPORT int syn_add_rmsnorm(float*, const float*, int, int, const int*, int, const void*, int, float, float, void*, int, int, hipStream_t);
SYN_EXPORT int syn_gemm(const void*, const void*, void*, int, int, int, int, int, int, int, int, int, int, float*, int64_t, hipStream_t);
SYN_EXPORT int64_t syn_gemm_f32_scratch(int, int, int);
SYN_EXPORT int syn_qk_norm_rope_kv_write(const void*, int, void*, void*, void*, int, const int*, int, const int*, const int*, const void*,
                                         const void*, int, float, float, const float*, const float*, int, int, int, int, int, int, hipStream_t);
SYN_EXPORT int syn_attention_f32(const float*, const float*, const float*, const int*, int, const int*, const int*, float*, float, int, int,
                                 int, int, int, const float*, float, int, hipStream_t);
SYN_EXPORT int syn_swiglu(const void*, void*, int, int, int, int, float, hipStream_t);

// The layer as the host hands it over: pointers and whole numbers as 64-bit words, in this order.
struct BlockF32 {
  float *resid, *delta, *out, *work;      // delta: what the residual has still to get (or null); work: syn_block_f32_floats
  void *gain1, *w_qkv, *q_gain, *k_gain, *cos_t, *sin_t, *k_pages, *v_pages;
  int *page_table, *tok_seq, *tok_pos;
  float* slopes;
  void *w_o, *gain2, *w_gate_up, *w_down;
  int64_t gain1_f32, qk_gain_f32, gain2_f32, table_stride, n, hidden, nh, nkv, hd, rot, window, write_kv, inner, act, prompts;
};

static int64_t block_piece(int64_t floats) { return (floats + 63) / 64 * 64; }
static int64_t block_rows(int64_t n, int64_t hidden, int64_t nh, int64_t hd) { return block_piece(n * (hidden > nh * hd ? hidden : nh * hd)); }
static int64_t block_wide(int64_t n, int64_t nh, int64_t nkv, int64_t hd, int64_t inner) {
  return block_piece(n * ((nh + 2 * nkv) * hd > 2 * inner ? (nh + 2 * nkv) * hd : 2 * inner));
}
static int64_t block_last(int64_t n, int64_t hidden, int64_t nh, int64_t hd, int64_t inner) {
  const int64_t rows = hidden > nh * hd ? hidden : nh * hd;
  return block_piece(n * (rows > inner ? rows : inner));
}
static int64_t block_products(int64_t n, int64_t hidden, int64_t nh, int64_t nkv, int64_t hd, int64_t inner) {
  return std::max({syn_gemm_f32_scratch((int)n, (int)((nh + 2 * nkv) * hd), (int)hidden), syn_gemm_f32_scratch((int)n, (int)hidden, (int)(nh * hd)),
                   syn_gemm_f32_scratch((int)n, (int)(2 * inner), (int)hidden), syn_gemm_f32_scratch((int)n, (int)hidden, (int)inner)});
}
// floats of working memory of a layer with n tokens
SYN_EXPORT int64_t syn_block_f32_floats(int64_t n, int64_t hidden, int64_t nh, int64_t nkv, int64_t hd, int64_t inner) {
  return block_rows(n, hidden, nh, hd) + block_wide(n, nh, nkv, hd, inner) + block_last(n, hidden, nh, hd, inner) +
         block_products(n, hidden, nh, nkv, hd, inner);
}

// reals: eps1, gain offset 1, q/k eps, q/k gain offset, scale, soft cap, eps2, gain offset 2, the activation's limit
SYN_EXPORT int syn_block_f32(const void* words, const double* reals, hipStream_t stream) {
  const BlockF32& b = *(const BlockF32*)words;
  const int n = (int)b.n, H = (int)b.hidden, nh = (int)b.nh, nkv = (int)b.nkv, hd = (int)b.hd, I = (int)b.inner;
  SYN_CHECK(b.n > 0 && b.n < (1 << 30) && H > 0 && nh > 0 && nkv > 0 && hd > 0 && I > 0, "block_f32: empty input");
  float* rows = b.work;                                        // a norm's rows, then attention's, then the second norm's
  float* wide = rows + block_rows(n, H, nh, hd);               // q, k, v; then gate and up
  float* last = wide + block_wide(n, nh, nkv, hd, I);          // queries; then the mixer's result; then the activation's
  float* products = last + block_last(n, H, nh, hd, I);        // the products' own
  const int64_t products_floats = block_products(n, H, nh, nkv, hd, I);
  int rc = syn_add_rmsnorm(b.resid, b.delta, 1, n, nullptr, n, b.gain1, (int)b.gain1_f32, (float)reals[1], (float)reals[0], rows, 1, H, stream);
  if (!rc) rc = syn_gemm(rows, b.w_qkv, wide, 0, n, (nh + 2 * nkv) * hd, H, 0, 1, 0, 0, -1, 0, products, products_floats, stream);
  if (!rc)
    rc = syn_qk_norm_rope_kv_write(wide, 0, last, b.k_pages, b.v_pages, 1, b.page_table, (int)b.table_stride, b.tok_seq, b.tok_pos, b.q_gain,
                                   b.k_gain, (int)b.qk_gain_f32, (float)reals[3], (float)reals[2], (const float*)b.cos_t,
                                   (const float*)b.sin_t, (int)b.rot, n, nh, nkv, hd, (int)b.write_kv, stream);
  if (!rc)
    rc = syn_attention_f32(last, (const float*)b.k_pages, (const float*)b.v_pages, b.page_table, (int)b.table_stride, b.tok_seq, b.tok_pos, rows,
                           (float)reals[4], (int)b.window, n, nh, nkv, hd, b.slopes, (float)reals[5], (int)b.prompts, stream);
  if (!rc) rc = syn_gemm(rows, b.w_o, last, 0, n, H, nh * hd, 0, 1, 0, 0, -1, 0, products, products_floats, stream);
  if (!rc) rc = syn_add_rmsnorm(b.resid, last, 1, n, nullptr, n, b.gain2, (int)b.gain2_f32, (float)reals[7], (float)reals[6], rows, 1, H, stream);
  if (!rc) rc = syn_gemm(rows, b.w_gate_up, wide, 0, n, 2 * I, H, 0, 1, 0, 0, -1, 0, products, products_floats, stream);
  if (!rc) rc = syn_swiglu(wide, last, 1, n, I, (int)b.act, (float)reals[8], stream);
  if (!rc) rc = syn_gemm(last, b.w_down, b.out, 0, n, H, I, 0, 1, 0, 0, -1, 0, products, products_floats, stream);
  return rc;
}
