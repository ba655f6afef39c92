// Attention over the paged cache in true 32-bit: four online softmaxes over blocks of 64 keys in turns.  Any
// head size up to 256, prefill and decode alike: one wave, or four, for each (token, head) with plain FMA; for prompts 16 (token,
// head) rows a workgroup on the matrix units, with the same bits.
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

// The same sums on the matrix units, for prompts: 16 (token, head) rows of one kv head a workgroup, a wave a class of blocks.
//   S^T (16 keys x 16 rows) = K . Q^T, O^T (16 dims x 16 rows) += V^T . P^T with v_mfma_f32_16x16x4_f32, whose sum over its four
// k-values is a chain of fused multiply-adds in their order (checked against such chains bit for bit, values below the normal range
// among them).  A lane loads 16 bytes and gives one value to each of four such instructions with sums of their own, which are the
// four chains of the kernel above, and what it holds of S^T is its share of P^T: a row's bits are those of that kernel, to which few
// tokens, windows and terms on the scores go.  (One chain in place of four: twice the error against 64 bits.)
// Where a value that a weight of zero meets may be no finite number (0 times which is no number), the block's weighted values are
// taken as above instead.  What bounds it: the loads' way (a wave's block is 32 KB of keys and as much of values, and 128 + 128
// matrix instructions, 3.4 us).  490 tokens of 120, 137 and 233 with 32 heads of 128 over 8: 228 -> 87 us; 480 tokens of
// one sequence 501 -> 122, 20 portions of 16 behind 400 477 -> 144, 600 tokens with 4 heads of 16 25 -> 13.
template <int DT>
__global__ void __launch_bounds__(256, 2)
attn_f32_tiles_kernel(const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
                      const int* __restrict__ page_table, int table_stride, const int* __restrict__ tok_seq,
                      const int* __restrict__ tok_pos, float* __restrict__ out, float scale, int n_tokens, int nh, int nkv) {
#pragma clang fp contract(off)
  constexpr int HD = 16 * DT, CLASSES = 4, T = SYN_PAGE / 16;
  __shared__ __attribute__((aligned(16))) float part[CLASSES][16][HD + 4];
  __shared__ float stat[CLASSES][16][2];
  __shared__ __attribute__((aligned(16))) float ps_all[CLASSES][SYN_PAGE][16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SYN_WAVE), lane = threadIdx.x % SYN_WAVE, r16 = lane % 16, g = lane / 16;
  const int G = nh / nkv, kvh = blockIdx.y, rows = n_tokens * G;
  const int row0 = (int)(gridDim.x - 1 - blockIdx.x) * 16;                // (late rows see the most keys and come first)
  const int flat = min(row0 + r16, rows - 1), tok = flat / G, head = kvh * G + flat % G;
  const int pos = tok_pos[tok];
  f32x4 qf[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) qf[t] = *(const f32x4*)(q + ((size_t)tok * nh + head) * HD + 16 * t + 4 * g);
  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int tok_last = min(row0 + 15, rows - 1) / G;
  for (int first = row0 / G; first <= tok_last;) {
    // the tokens first .. end - 1 of one sequence; rows of other tokens see nothing meanwhile, which leaves them as they are
    const int seq = __builtin_amdgcn_readfirstlane(tok_seq[first]);
    int end = first, top = 0;
    while (end <= tok_last && tok_seq[end] == seq) top = max(top, tok_pos[end]), ++end;
    top = __builtin_amdgcn_readfirstlane(top), end = __builtin_amdgcn_readfirstlane(end);
    const int seen = tok >= first && tok < end ? pos : -1;
    first = end;
    for (int kb = wave; kb <= top / SYN_PAGE; kb += CLASSES) {
      const int page = page_table[(size_t)seq * table_stride + kb];
      const size_t base = ((size_t)page * nkv + kvh) * SYN_PAGE * HD;
      const float* kp = k_pages + base + (size_t)r16 * HD + 4 * g;
      const float* vp = v_pages + base + (size_t)r16 * SYN_PAGE + 4 * g;
      f32x4 s[T], of[4][T];      // (a chain for each of the four neighbours, as above)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < T; ++t) of[e][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        f32x4 kf[T];
#pragma unroll
        for (int t = 0; t < T; ++t) kf[t] = *(const f32x4*)(kp + (size_t)16 * t * HD + 16 * d);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < T; ++t) of[e][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][e], qf[d][e], of[e][t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < T; ++t) s[t] = (of[0][t] + of[1][t]) + (of[2][t] + of[3][t]);
      // s[t][e]: key kb * 64 + 16 t + 4 g + e against the lane's row
      float most = -INFINITY;
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[t][e] = kb * SYN_PAGE + 16 * t + 4 * g + e <= seen ? s[t][e] * scale : -INFINITY;
          most = fmaxf(most, s[t][e]);
        }
      most = fmaxf(most, __shfl_xor(most, 16, SYN_WAVE));
      most = fmaxf(most, __shfl_xor(most, 32, SYN_WAVE));
      const float m_new = fmaxf(m, most);
      const float alpha = m == m_new ? 1.f : expf(m - m_new);
      float u[4];
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t][e] = s[t][e] == -INFINITY ? 0.f : expf(s[t][e] - m_new);
      // (the order of a sum over a wave's 64 lanes, a key a lane)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        u[e] = (s[0][e] + s[2][e]) + (s[1][e] + s[3][e]);
        u[e] += __shfl_xor(u[e], 32, SYN_WAVE);
        u[e] += __shfl_xor(u[e], 16, SYN_WAVE);
      }
      l = fmaf(l, alpha, (u[0] + u[2]) + (u[1] + u[3]));
      m = m_new;
      const int left = top - kb * SYN_PAGE;          // slots behind it may hold anything: taken as zeros
      float strange = 0.f;                           // NaN where some value is infinite or no number
      f32x4 before[DT];
#pragma unroll
      for (int d = 0; d < DT; ++d) before[d] = o[d] * alpha;
      constexpr int DG = DT % 4 == 0 ? 4 : DT % 3 == 0 ? 3 : DT % 2 == 0 ? 2 : DT == 1 || DT > 7 ? 1 : DT;      // tiles of dims at a time
#pragma unroll
      for (int d0 = 0; d0 < DT; d0 += DG) {
        f32x4 sum[DG][4];
#pragma unroll
        for (int d = 0; d < DG; ++d) {
          sum[d][0] = before[d0 + d];
#pragma unroll
          for (int e = 1; e < 4; ++e) sum[d][e] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
          f32x4 vf[DG];
#pragma unroll
          for (int d = 0; d < DG; ++d) vf[d] = *(const f32x4*)(vp + (size_t)16 * (d0 + d) * SYN_PAGE + 16 * t);
          if (left < 16 * t + 15) {
#pragma unroll
            for (int d = 0; d < DG; ++d)
#pragma unroll
              for (int e = 0; e < 4; ++e) vf[d][e] = 16 * t + 4 * g + e <= left ? vf[d][e] : 0.f;
          }
#pragma unroll
          for (int d = 0; d < DG; ++d)
#pragma unroll
            for (int e = 0; e < 4; ++e) strange = fmaf(vf[d][e], 0.f, strange);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < DG; ++d) sum[d][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[d][e], s[t][e], sum[d][e], 0, 0, 0);
        }
#pragma unroll
        for (int d = 0; d < DG; ++d) o[d0 + d] = (sum[d][0] + sum[d][1]) + (sum[d][2] + sum[d][3]);
      }
      if (__any(strange != strange)) {
        float(*ps)[16] = ps_all[wave];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) ps[16 * t + 4 * g + e][r16] = s[t][e];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float* vr = v_pages + base + (size_t)(16 * d + 4 * g + i) * SYN_PAGE;
            f32x4 a4 = {before[d][i], 0.f, 0.f, 0.f};
            for (int j = 0; j < SYN_PAGE; j += 4)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float p = ps[j + e][r16];
                a4[e] = fmaf(p, p != 0.f ? vr[j + e] : 0.f, a4[e]);
              }
            o[d][i] = (a4[0] + a4[1]) + (a4[2] + a4[3]);
          }
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  // o[d][e]: dim 16 d + 4 g + e of the lane's row; the classes together as above
#pragma unroll
  for (int d = 0; d < DT; ++d) *(f32x4*)&part[wave][r16][16 * d + 4 * g] = o[d];
  if (g == 0) stat[wave][r16][0] = m, stat[wave][r16][1] = l;
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * HD; i += 256) {
    const int r = i / HD, d = i % HD;
    if (row0 + r >= rows) continue;
    float top = stat[0][r][0], sum = 0.f, f[CLASSES], v = 0.f;
#pragma unroll
    for (int c = 1; c < CLASSES; ++c) top = fmaxf(top, stat[c][r][0]);
#pragma unroll
    for (int c = 0; c < CLASSES; ++c) {
      f[c] = stat[c][r][0] == -INFINITY ? stat[c][r][1] : expf(stat[c][r][0] - top);
      sum = fmaf(f[c], stat[c][r][1], sum);
    }
#pragma unroll
    for (int c = 0; c < CLASSES; ++c)
      if (f[c] != 0.f) v = fmaf(f[c], part[c][r][d], v);
    out[((size_t)((row0 + r) / G) * nh + kvh * G + (row0 + r) % G) * HD + d] = v / sum;
  }
}

// slopes [nh] float or null, softcap (0: none): see ScoreTerms; prompts: 16 rows a workgroup may take the step (the host's rule, which
// knows the lengths: a workgroup walks the sequences of its rows one after another, ops.prompt_rows_pay)
SYN_EXPORT int syn_attention_f32(const float* q, const float* k_pages, const float* v_pages, const int* page_table,
                                 int table_stride, const int* tok_seq, const int* tok_pos, float* out, float scale,
                                 int window, int n_tokens, int nh, int nkv, int hd, const float* slopes, float softcap,
                                 int prompts, hipStream_t stream) {
  SYN_CHECK(softcap >= 0.f, "attention_f32: a soft cap of %g", (double)softcap);
  SYN_CHECK(n_tokens > 0 && nh > 0 && nkv > 0, "attention_f32: empty input");
  SYN_CHECK(nh % nkv == 0, "attention_f32: %d heads do not divide into %d kv heads", nh, nkv);
  SYN_CHECK(hd > 0 && hd <= ATTN32_MAX_HD, "attention_f32: head size %d is outside 1..%d", hd, ATTN32_MAX_HD);
  const ScoreTerms terms = {slopes, softcap};
  const bool aligned = (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0;
  const bool vec = hd % 4 == 0 && aligned;
  // beyond eight waves a compute unit of (token, head) rows (70 tokens, 32 heads of 128: 28 us a wave a row, 25 so; below, keys over waves)
  if (prompts && hd % 16 == 0 && aligned && hd <= 128 && window <= 0 && !slopes && softcap == 0.f && (uintptr_t)q % 16 == 0 &&
      (long)n_tokens * nh > 8L * syn_compute_units() && nkv <= 65535) {
    const dim3 grid((unsigned)(((long)n_tokens * (nh / nkv) + 15) / 16), nkv);
#define SYN_ATTN32_TILES(DT)                                                                                                        \
  case DT:                                                                                                                          \
    attn_f32_tiles_kernel<DT><<<grid, 256, 0, stream>>>(q, k_pages, v_pages, page_table, table_stride, tok_seq, tok_pos, out, scale, \
                                                        n_tokens, nh, nkv);                                                         \
    break;
    switch (hd / 16) {
      SYN_ATTN32_TILES(1) SYN_ATTN32_TILES(2) SYN_ATTN32_TILES(3) SYN_ATTN32_TILES(4) SYN_ATTN32_TILES(5) SYN_ATTN32_TILES(6)
      SYN_ATTN32_TILES(7) SYN_ATTN32_TILES(8)
    }
#undef SYN_ATTN32_TILES
    SYN_LAUNCH_CHECK("attention_f32_tiles");
    return 0;
  }
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
