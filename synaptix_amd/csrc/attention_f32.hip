// Attention over the paged cache in true 32-bit: one wave, or four, for each (token, head), plain FMA,
// four online softmaxes over blocks of 64 keys in turns.  Any head size up to 256, prefill and decode alike.
//
//   query of token t sits at position p = tok_pos[t] of sequence tok_seq[t];
//   key j is visible iff j <= p and (window <= 0 or j > p - window);
//   head h reads kv head h / (nh / nkv).
// Definition as in crates/synaptix-kernels-cuda/tests/cuda_flash_decode.rs:32-90 and the mask of
// crates/synaptix-models/llm/common/src/model.rs:2581-2596.
//
// Cache pages hold 64 tokens: k_pages[page, kv_head, token, d], v_pages[page, kv_head, d, token].
#include "common.h"

#define ATTN32_MAX_HD 256

// (16 bytes that start at any float: one load all the same)
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// The blocks of keys of a (token, head) fall into four classes in turns, each with a running softmax of its own, merged in the order
// of the classes.  WAVES waves a workgroup.  SPLIT: a wave a class (few tokens: a wave alone would walk a sequence's keys one block
// after another); else each wave has a head of its own and takes the classes one after another, the heads of one kv head
// side by side, which then share its keys and values in the compute unit's cache.  The sums are the same either way: a
// token's result does not depend on how many others are in the step.
// A lane has a key's row, then a dimension's row, to itself: 16 bytes at a time each 128-byte line is asked for 8 times instead of
// 32.  The values' rows (64 floats) are always read so, keys and queries where the head size is a multiple of 4 (VEC).  490 tokens of
// 120, 137 and 233 with 32 heads of 128 over 8: 839 -> 265 us.  Values one at a time behind a branch on their weight: three
// times 400 tokens with 7 heads of 63 take 809 us, so 424.
template <int WAVES, bool SPLIT, bool VEC>
__global__ void __launch_bounds__(WAVES * SYN_WAVE)
attn_f32_kernel(const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
                const int* __restrict__ page_table, int table_stride, const int* __restrict__ tok_seq,
                const int* __restrict__ tok_pos, float* __restrict__ out, float scale, int window, int nh, int nkv,
                int hd, ScoreTerms terms) {
#pragma clang fp contract(off)      // (fused where it says so, the same in every variant)
  __shared__ __attribute__((aligned(16))) float qs_all[WAVES][ATTN32_MAX_HD];
  __shared__ __attribute__((aligned(16))) float ps_all[WAVES][SYN_PAGE];
  constexpr int CLASSES = 4;
  static_assert(!SPLIT || WAVES == CLASSES, "a wave a class");
  __shared__ float part_all[SPLIT ? 1 : WAVES][CLASSES][ATTN32_MAX_HD], stat_all[SPLIT ? 1 : WAVES][CLASSES][2];
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  const int tok = blockIdx.x, head = SPLIT ? (int)blockIdx.y : (int)blockIdx.y * WAVES + wave;
  float* qs = qs_all[wave];
  float* ps = ps_all[wave];
  const int seq = tok_seq[tok], pos = tok_pos[tok];
  const int kvh = head / (nh / nkv);
  const float* qr = q + ((size_t)tok * nh + head) * hd;
  for (int d = lane; d < hd; d += SYN_WAVE) qs[d] = qr[d];
  // (a wave writes and reads its own part of LDS only: what it wrote is there for its own later reads)
  __builtin_amdgcn_wave_barrier();

  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const bool with_terms = score_terms_on(terms);
  const float slope = terms.slopes ? terms.slopes[head] : 0.f;
  auto part = part_all[SPLIT ? 0 : wave];
  auto stat = stat_all[SPLIT ? 0 : wave];
  for (int c = SPLIT ? wave : 0; c < (SPLIT ? wave + 1 : CLASSES); ++c) {
    float m = -INFINITY, l = 0.f;
    float o[ATTN32_MAX_HD / SYN_WAVE] = {0.f, 0.f, 0.f, 0.f};
    for (int kb = lo / SYN_PAGE + c; kb <= pos / SYN_PAGE; kb += CLASSES) {
      const int page = page_table[(size_t)seq * table_stride + kb];
      const size_t base = ((size_t)page * nkv + kvh) * SYN_PAGE * hd;
      const int key = kb * SYN_PAGE + lane;
      const bool valid = key >= lo && key <= pos;
      float s = -INFINITY;
      if (valid) {
        const float* kr = k_pages + base + (size_t)lane * hd;
        float dot = 0.f;
        if constexpr (VEC) {
          f32x4 d4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
          for (int d = 0; d < hd; d += 4) {
            const f32x4 kk = *(const f32x4*)(kr + d), qq = *(const f32x4*)(qs + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) d4[e] = fmaf(qq[e], kk[e], d4[e]);
          }
          dot = (d4[0] + d4[1]) + (d4[2] + d4[3]);
        } else {
          for (int d = 0; d < hd; ++d) dot = fmaf(qs[d], kr[d], dot);
        }
        s = dot * scale;
        if (with_terms) s = score_with_terms(s, slope, terms.softcap, pos, key);
      }
      // (a score of -inf weighs nothing, also among none but such; one that is no number stays one in p and l)
      const float m_new = fmaxf(m, wave_max(s));
      const float alpha = m == m_new ? 1.f : expf(m - m_new);
      const float p = s == -INFINITY ? 0.f : expf(s - m_new);
      l = fmaf(l, alpha, wave_sum(p));
      m = m_new;
      ps[lane] = p;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < ATTN32_MAX_HD / SYN_WAVE; ++i) {
        const int d = lane + i * SYN_WAVE;
        if (d < hd) {
          const float* vr = v_pages + base + (size_t)d * SYN_PAGE;
          // (slots past the sequence's end may hold anything: a weight of zero takes nothing from them)
          f32x4 a4 = {o[i] * alpha, 0.f, 0.f, 0.f};
#pragma unroll 8
          for (int j = 0; j < SYN_PAGE; j += 4) {
            const f32x4 vv = *(const f32x4_any*)(vr + j), pp = *(const f32x4*)(ps + j);
#pragma unroll
            for (int e = 0; e < 4; ++e) a4[e] = fmaf(pp[e], pp[e] != 0.f ? vv[e] : 0.f, a4[e]);
          }
          o[i] = (a4[0] + a4[1]) + (a4[2] + a4[3]);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) stat[c][0] = m, stat[c][1] = l;
#pragma unroll
    for (int i = 0; i < ATTN32_MAX_HD / SYN_WAVE; ++i) {
      const int d = lane + i * SYN_WAVE;
      if (d < hd) part[c][d] = o[i];
    }
  }
  // the common maximum first, then sums in the order of the classes (one without a weight has m = -inf and l = 0, or an l that is
  // no number where a score was none)
  if constexpr (SPLIT) {
    __syncthreads();
    if (wave != 0) return;
  } else {
    __builtin_amdgcn_wave_barrier();
  }
  float top = stat[0][0], l = 0.f, f[CLASSES], o[ATTN32_MAX_HD / SYN_WAVE];
#pragma unroll
  for (int c = 1; c < CLASSES; ++c) top = fmaxf(top, stat[c][0]);
#pragma unroll
  for (int c = 0; c < CLASSES; ++c) {
    f[c] = stat[c][0] == -INFINITY ? stat[c][1] : expf(stat[c][0] - top);
    l = fmaf(f[c], stat[c][1], l);
  }
#pragma unroll
  for (int i = 0; i < ATTN32_MAX_HD / SYN_WAVE; ++i) {
    const int d = lane + i * SYN_WAVE;
    o[i] = 0.f;
#pragma unroll
    for (int c = 0; c < CLASSES; ++c)
      if (d < hd && f[c] != 0.f) o[i] = fmaf(f[c], part[c][d], o[i]);
  }
  float* orow = out + ((size_t)tok * nh + head) * hd;
#pragma unroll
  for (int i = 0; i < ATTN32_MAX_HD / SYN_WAVE; ++i) {
    const int d = lane + i * SYN_WAVE;
    if (d < hd) orow[d] = o[i] / l;
  }
}

// slopes [nh] float or null, softcap (0: none): see ScoreTerms
SYN_EXPORT int syn_attention_f32(const float* q, const float* k_pages, const float* v_pages, const int* page_table,
                                 int table_stride, const int* tok_seq, const int* tok_pos, float* out, float scale,
                                 int window, int n_tokens, int nh, int nkv, int hd, const float* slopes, float softcap,
                                 hipStream_t stream) {
  SYN_CHECK(softcap >= 0.f, "attention_f32: a soft cap of %g", (double)softcap);
  SYN_CHECK(n_tokens > 0 && nh > 0 && nkv > 0, "attention_f32: empty input");
  SYN_CHECK(nh % nkv == 0, "attention_f32: %d heads do not divide into %d kv heads", nh, nkv);
  SYN_CHECK(hd > 0 && hd <= ATTN32_MAX_HD, "attention_f32: head size %d is outside 1..%d", hd, ATTN32_MAX_HD);
  const ScoreTerms terms = {slopes, softcap};
  const bool vec = hd % 4 == 0 && (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0;
#define SYN_ATTN32(WAVES, SPLIT)                                                                                              \
  (vec ? attn_f32_kernel<WAVES, SPLIT, true> : attn_f32_kernel<WAVES, SPLIT, false>)                                          \
      <<<dim3(n_tokens, SPLIT ? nh : nh / WAVES), WAVES * SYN_WAVE, 0, stream>>>(q, k_pages, v_pages, page_table, table_stride, \
                                                                                tok_seq, tok_pos, out, scale, window, nh, nkv, hd, terms)
  // up to eight waves a compute unit: the waves of a workgroup split the keys; beyond them the chip is full without
  if ((long)n_tokens * nh <= 8L * syn_compute_units()) SYN_ATTN32(4, true);
  else if ((nh / nkv) % 4 == 0) SYN_ATTN32(4, false);
  else if ((nh / nkv) % 2 == 0) SYN_ATTN32(2, false);
  else SYN_ATTN32(1, false);
#undef SYN_ATTN32
  SYN_LAUNCH_CHECK("attention_f32");
  return 0;
}
