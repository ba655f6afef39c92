// Latent attention in bf16 on the matrix cores: every head's query against ONE key row a cached token.
//
//   q       [N][heads][R]        R = rank + rot: the query in the latent's space, then its rotated part
//   k_pages [pages][64][R]       a token's row [latent | rotated key part]
//   v_pages [pages][rank x 64]   the latent once more, in the order of this kernel's fragments (la_v_offset): the
//                                8 values that a lane feeds into one matrix instruction lie together, a wave's 64
//                                lanes one after another: a fragment is 1 KB of consecutive bytes
//   out     [N][heads][rank]     sum_j softmax_j(scale q . k_j) k_j[:rank]  over the keys j that the query sees:
//                                j <= position, and position - j < window if there is a window
//
// Since all heads share the keys, the 16 rows of a tile are 16 consecutive (token, head) pairs of one sequence: for
// a single token its heads (decoding is a small matrix product, not a matrix-vector one), for a prompt a few tokens
// with all their heads:
//   S^T (keys x rows)  = K (16 keys x k) . Q^T (k x 16 rows)        a lane holds four keys of ONE row
//   O^T (rank x rows) += V^T (16 values x 32 keys) . P^T (32 keys x 16 rows)
// and what a lane holds of S^T is exactly its share of the operand P^T (the 32 keys of a k-step are taken in the
// order in which two score tiles leave them, and V^T's 8-byte pieces are fetched in that order too).  The scores
// and weights are 32-bit; a weight meets V as two bf16 numbers (the weight rounded, and what the rounding left), so
// it counts with 16 bits of mantissa although the product runs in bf16; sums are 32-bit.
// The four waves of a workgroup work on the same rows, with a quarter of a page's keys and of the values each.  Few tiles
// (single tokens) take a workgroup each and their pages may be cut into splits (grid y) whose partial results a second
// kernel merges; many tiles (prompts) go four to a workgroup.
#include "common.h"

#define LA_ROWS 16

template <bool X32> struct LaFrag;
template <> struct LaFrag<false> { typedef bf16x4 type; };
template <> struct LaFrag<true> { typedef bf16x8 type; };

__device__ __forceinline__ f32x4 la_mfma(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4_t, a), __builtin_bit_cast(short4_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 la_mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Where value d of the token in slot `slot` of a page lies in a bf16 value page of latent attention: fragment (d / 16,
// slot / 32), lane 16 g + d % 16, element e, with the 32 slots of a half in the order in which two tiles of scores
// leave them in a lane: e < 4: slot 4 g + e; e >= 4: slot 16 + 4 g + (e - 4).
__host__ __device__ __forceinline__ int la_v_offset(int d, int slot) {
  const int half = slot >> 5, s = slot & 31, second = s >> 4, g = (s & 15) >> 2, e = (s & 3) + 4 * second;
  return ((((d >> 4) * 2 + half) * 64 + g * 16 + (d & 15)) << 3) + e;
}

// the sequence and the unit inside it of global unit t, a unit being `unit_rows` consecutive (token, head) rows.
// Every wave searches for itself, 64 sequences at a time: a lane a sequence, a prefix sum of their units across the
// lanes, the first lane whose sum passes t (one trip to memory for 64 sequences, not one for each).  t is the same in
// all lanes of the wave.
__device__ __forceinline__ bool la_find_unit(int t, int unit_rows, const int* seq_start, int n_seqs, int nh, int& seq,
                                             int& unit, int& start, int& rows) {
  const int lane = threadIdx.x % SYN_WAVE;
  for (int b0 = 0; b0 < n_seqs; b0 += SYN_WAVE) {
    const int b = b0 + lane;
    const int s0 = b < n_seqs ? seq_start[b] : 0;
    const int n = b < n_seqs ? (seq_start[b + 1] - s0) * nh : 0;
    const int units = (n + unit_rows - 1) / unit_rows;
    int upto = units;                                    // units of the sequences b0 .. b
#pragma unroll
    for (int off = 1; off < SYN_WAVE; off <<= 1) {
      const int other = __shfl_up(upto, off, SYN_WAVE);
      if (lane >= off) upto += other;
    }
    const unsigned long long found = __ballot(t < upto);
    if (found) {
      const int at = __ffsll((long long)found) - 1;
      seq = b0 + at;
      unit = t - (__shfl(upto, at, SYN_WAVE) - __shfl(units, at, SYN_WAVE));
      start = __shfl(s0, at, SYN_WAVE);
      rows = __shfl(n, at, SYN_WAVE);
      return true;
    }
    t -= __shfl(upto, SYN_WAVE - 1, SYN_WAVE);
  }
  return false;
}

// Single tokens: a workgroup takes one tile; on every page its four waves split the keys for the scores and the values for
// the second product.
// DT: tiles of 16 values that the accumulators of the four waves hold (rank <= 16 DT); QS: k-steps that the query's registers
// hold (R <= QS * (X32 ? 32 : 16)); X32: k-steps of 32 (R a multiple of 32) or of 16.
template <int DT, int QS, bool X32>
__global__ void __launch_bounds__(256)
latent_attention_bf16_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
                             const int* __restrict__ page_table, int table_stride, const int* __restrict__ seq_start,
                             const int* __restrict__ seq_past, int n_seqs, bf16* __restrict__ out,
                             float* __restrict__ part_o, float* __restrict__ part_ml, float scale, int nh, int rank, int R,
                             int window, int n_splits) {
  typedef typename LaFrag<X32>::type frag;
  constexpr int KS = X32 ? 32 : 16, PIECE = KS / 4;
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE, i = lane % 16, g = lane / 16;
  const int split = blockIdx.y;
  int seq, unit, start, rows;
  if (!la_find_unit(blockIdx.x, LA_ROWS, seq_start, n_seqs, nh, seq, unit, start, rows)) return;
  const int past = seq_past[seq];
  const int flat0 = unit * LA_ROWS, flat_last = min(flat0 + LA_ROWS, rows) - 1;
  const bool row_ok = flat0 + i < rows;
  const int flat = row_ok ? flat0 + i : flat_last;       // a row beyond the tile's end repeats the last one, unstored
  const int tok = flat / nh, head = flat % nh, pos = past + tok;
  const int kv_len = past + rows / nh;
  // the pages that some row of the tile sees
  const int pos_lo = past + flat0 / nh, pos_hi = past + flat_last / nh;
  const int my_lo = (window > 0 ? max(0, pos_lo - window + 1) : 0) / SYN_PAGE, my_hi = pos_hi / SYN_PAGE;
  const int n_qs = R / KS, n_dt = rank / 16;

  frag qf[QS];
  const bf16* qrow = q + ((size_t)(start + tok) * nh + head) * R + g * PIECE;
#pragma unroll
  for (int ks = 0; ks < QS; ++ks)
    if (ks < n_qs) qf[ks] = *(const frag*)(qrow + ks * KS);

  // a wave holds a quarter of the value tiles (DTW of them, from dt0 on)
  constexpr int DTW = DT / 4;
  const int dt0 = wave * ((n_dt + 3) / 4), dt_end = min(dt0 + (n_dt + 3) / 4, n_dt);
  f32x4 acc[DTW];
#pragma unroll
  for (int dt = 0; dt < DTW; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int* pages = page_table + (size_t)seq * table_stride;

  // This split's share of the tile's pages, one after another, the four waves on the same page: wave w multiplies
  // the 16 keys w * 16 .. of the page with the queries, the waves exchange maxima, sums and weights through LDS (the
  // weights already in the order of the second product's operand), and wave w then multiplies its quarter of the
  // value tiles with all 64 weights.  Every load of a phase is asked for before the first result is needed, the
  // values before the scores are exchanged.  What goes through LDS is kept twice, for pages in turns: two barriers
  // a page are enough.
  __shared__ float sh_max[2][4][LA_ROWS], sh_sum[2][4][LA_ROWS];
  __shared__ __attribute__((aligned(16))) bf16 sh_hi[2][2][SYN_WAVE][8], sh_lo[2][2][SYN_WAVE][8];
  const int chunk = (my_hi - my_lo + n_splits) / n_splits;
  const int p0 = my_lo + split * chunk, p1 = min(p0 + chunk, my_hi + 1);
  int par = 0;
  for (int p = p0; p < p1; ++p, par ^= 1) {
    const int page = pages[p];
    const bf16* kb = k_pages + (size_t)page * SYN_PAGE * R + (size_t)(wave * 16 + i) * R + g * PIECE;
    const bf16* vb = v_pages + (size_t)page * rank * SYN_PAGE + lane * 8;
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < QS; ++ks)
      if (ks < n_qs) s = la_mfma(*(const frag*)(kb + ks * KS), qf[ks], s);
    bf16x8 va[DTW][2];
#pragma unroll
    for (int j = 0; j < DTW; ++j)
      if (dt0 + j < dt_end) {
        va[j][0] = *(const bf16x8*)(vb + ((dt0 + j) * 2) * 512);
        va[j][1] = *(const bf16x8*)(vb + ((dt0 + j) * 2 + 1) * 512);
      }
    // s[e]: key p * 64 + wave * 16 + 4 g + e against this lane's row
    const int key0 = p * SYN_PAGE + wave * 16 + 4 * g;
    float top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int key = key0 + e;
      const bool seen = key <= pos && (window <= 0 || pos - key < window);
      s[e] = seen ? s[e] * scale : -INFINITY;
      top = fmaxf(top, s[e]);
    }
    top = fmaxf(top, __shfl_xor(top, 16, SYN_WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, SYN_WAVE));
    if (g == 0) sh_max[par][wave][i] = top;
    __syncthreads();
    float m_new = m;
#pragma unroll
    for (int w = 0; w < 4; ++w) m_new = fmaxf(m_new, sh_max[par][w][i]);
    const float base = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = expf(m - base);
    float sum = 0.f;
    bf16x4 hi, lo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float w = expf(s[e] - base);
      sum += w;
      hi[e] = (bf16)w;
      lo[e] = (bf16)(w - (float)hi[e]);
    }
    sum += __shfl_xor(sum, 16, SYN_WAVE);
    sum += __shfl_xor(sum, 32, SYN_WAVE);
    if (g == 0) sh_sum[par][wave][i] = sum;
    // key tile `wave` is elements 4 (wave % 2) .. of the operand of half wave / 2
    *(bf16x4*)&sh_hi[par][wave >> 1][lane][4 * (wave & 1)] = hi;
    *(bf16x4*)&sh_lo[par][wave >> 1][lane][4 * (wave & 1)] = lo;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) total += sh_sum[par][w][i];
    l = l * alpha + total;
    m = m_new;
    const int left = kv_len - p * SYN_PAGE;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bf16x8 ph = *(const bf16x8*)&sh_hi[par][half][lane][0], pl = *(const bf16x8*)&sh_lo[par][half][lane][0];
#pragma unroll
      for (int j = 0; j < DTW; ++j)
        if (dt0 + j < dt_end) {
          if (half == 0) acc[j] *= alpha;
          bf16x8 a = va[j][half];
          if (left < SYN_PAGE) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (32 * half + 4 * g + e >= left) a[e] = (bf16)0.f;
              if (32 * half + 16 + 4 * g + e >= left) a[4 + e] = (bf16)0.f;
            }
          }
          acc[j] = la_mfma(a, ph, acc[j]);
          acc[j] = la_mfma(a, pl, acc[j]);
        }
    }
  }
  // acc[j][e]: value (dt0 + j) * 16 + 4 g + e of this lane's row
  if (n_splits == 1) {
    if (!row_ok) return;
    const float inv = 1.f / l;
    bf16* orow = out + ((size_t)(start + tok) * nh + head) * rank + 4 * g;
#pragma unroll
    for (int j = 0; j < DTW; ++j)
      if (dt0 + j < dt_end) {
        bf16x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = (bf16)(acc[j][e] * inv);
        *(bf16x4*)(orow + (dt0 + j) * 16) = r;
      }
  } else {
    // (blockIdx.x is the tile's number among all tiles)
    const size_t at = ((size_t)blockIdx.x * n_splits + split) * LA_ROWS + i;
    if (g == 0 && wave == 0) part_ml[2 * at] = m, part_ml[2 * at + 1] = l;
    float* prow = part_o + at * rank + 4 * g;
#pragma unroll
    for (int j = 0; j < DTW; ++j)
      if (dt0 + j < dt_end) *(f32x4*)(prow + (dt0 + j) * 16) = acc[j];
  }
}

// ---------------------------------------------------------------- prompts: 64 (token, head) rows a workgroup
// The four waves of a workgroup work on the same 64 rows: for the scores a wave takes the 16 keys w * 16 .. of a page, for the
// second product a quarter of the value tiles, so each piece of keys and values goes to one wave, straight from memory into its
// registers, and is used for four tiles of rows.  The queries are what all waves share: their first QR k-steps stay in
// registers, the others in LDS in the order of the fragments; weights meet in LDS as above.  A page's values are on their way
// during its scores, the next page's keys during its second product.
// A page is 72 + 128 matrix instructions a wave with rows of 512 + 64 values, a quarter of what it takes: the phases follow
// each other with one wave a SIMD (scores, weights, their exchange, second product), and 140 KB a page come from L2.  Against a
// wave a tile of 16 rows with the page staged through LDS between two barriers, every load waited for: 1,500 tokens, 32 heads,
// 627 -> 218 us; eight sequences, 3,270 tokens in all: 584 -> 240 us.  Other rows, the same 1,500 tokens: 128 + 16 values 138 -> 52 us,
// 128 + 64 163 -> 119, 256 + 32 240 -> 122, 256 + 64 258 -> 127, 512 + 16 713 -> 221, 512 + 128 671 -> 237; 128 tokens behind 4,096 with
// 128 + 16 260 -> 121, 512 + 128 1,130 -> 323.
// The matrix instructions stand as inline assembly to keep the accumulators in vector registers and the fragments in the
// accumulation registers (left to itself the compiler moves 128 of them back and forth on every page, or spills); it does not
// know them for what they are, so their results are waited for by hand.
// The sums of a row are rescaled only where its maximum has grown by more than LA_LAZY since the last time: weights of up to
// 2^LA_LAZY are as exact as those of up to 1, and most pages need no pass over the accumulators.
// A sequence's last rows see the most pages and come first.
#define LA_LAZY 11.f
// the lanes l, l ^ 16, l ^ 32 and l ^ 48 together
template <typename F>
__device__ __forceinline__ float across16(float x, F of) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const unsigned a0 = a[0], a1 = a[1];
  const float y = of(__uint_as_float(a0), __uint_as_float(a1));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  const unsigned b0 = b[0], b1 = b[1];
  return of(__uint_as_float(b0), __uint_as_float(b1));
}
// DTW: value tiles of a wave (rank <= 64 DTW); QS: k-steps of 32 (R <= 32 QS; WHOLE: R = 32 QS)
template <int DTW, int QS, bool WHOLE>
__global__ void __launch_bounds__(256, 1)
latent_prompt_bf16_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
                          const int* __restrict__ page_table, int table_stride, const int* __restrict__ seq_start,
                          const int* __restrict__ seq_past, int n_seqs, bf16* __restrict__ out, float scale, int nh, int rank,
                          int R, int window) {
  constexpr int RT = 4, QR = QS < 8 ? QS : 8, QL = QS - QR;      // tiles of rows; k-steps of the queries in registers, in LDS
  __shared__ __attribute__((aligned(16))) bf16 q_lds[QL ? QL : 1][RT][SYN_WAVE][8];
  __shared__ __attribute__((aligned(16))) bf16 p_lds[2][2][RT][SYN_WAVE][8];      // [rounded, rest][half of the page]
  __shared__ __attribute__((aligned(16))) float max_lds[RT * 16][4];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SYN_WAVE), lane = threadIdx.x % SYN_WAVE, i = lane % 16, g = lane / 16;
  int seq, unit, start, rows;
  if (!la_find_unit(blockIdx.x, RT * LA_ROWS, seq_start, n_seqs, nh, seq, unit, start, rows)) return;
  seq = __builtin_amdgcn_readfirstlane(seq), start = __builtin_amdgcn_readfirstlane(start);
  rows = __builtin_amdgcn_readfirstlane(rows);
  unit = (rows + RT * LA_ROWS - 1) / (RT * LA_ROWS) - 1 - __builtin_amdgcn_readfirstlane(unit);
  const int past = seq_past[seq], kv_len = past + rows / nh;
  const int first = unit * RT * LA_ROWS, last = min(first + RT * LA_ROWS, rows) - 1;
  const int p_lo = (window > 0 ? max(0, past + first / nh - window + 1) : 0) / SYN_PAGE, p_hi = (past + last / nh) / SYN_PAGE;
  const size_t row0 = (size_t)start * nh;
  int pos[RT], unseen[RT];                        // (a row beyond the end repeats the last one, unstored)
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    pos[t] = past + min(first + t * 16 + i, last) / nh;
    unseen[t] = window > 0 ? pos[t] - window : -1;      // the row sees the keys behind this one, up to its own
  }

  const int seen_by_all = past + first / nh, unseen_by_some = window > 0 ? past + last / nh - window : -1;
  scale *= 1.4426950408889634f;

  const bf16x8 zero = {};
  auto query = [&](int ks, int t) {
    const int k = ks * 32 + g * 8;
    return WHOLE || k < R ? *(const bf16x8*)(q + (row0 + min(first + t * 16 + i, last)) * R + k) : zero;
  };
  bf16x8 qf[QR][RT];
#pragma unroll
  for (int ks = 0; ks < QR; ++ks)
#pragma unroll
    for (int t = 0; t < RT; ++t) qf[ks][t] = query(ks, t);
#pragma unroll
  for (int ks = 0; ks < QL; ++ks) *(bf16x8*)&q_lds[ks][wave][lane][0] = query(QR + ks, wave);

  const int n_dt = rank / 16;
  const int* pages = page_table + (size_t)seq * table_stride;
  bf16x8 kf[QS], vf[DTW][2];
  const unsigned k_at = (unsigned)((wave * 16 + i) * R + g * 8) * sizeof(bf16), v_at = (unsigned)(wave * DTW * 1024 + lane * 8) * sizeof(bf16);
  auto load_keys = [&](int page) {
    const BufferView v = buffer_view(k_pages + (size_t)page * SYN_PAGE * R, (size_t)SYN_PAGE * R * sizeof(bf16));
#pragma unroll
    for (int ks = 0; ks < QS; ++ks) kf[ks] = buffer_load16(v, WHOLE || ks * 32 + g * 8 < R ? k_at + ks * 64 : SYN_NOWHERE);
  };
  // (tiles behind the last one lie behind the view: zeros)
  auto load_values = [&](int page) {
    const BufferView v = buffer_view(v_pages + (size_t)page * SYN_PAGE * rank, (size_t)SYN_PAGE * rank * sizeof(bf16));
#pragma unroll
    for (int j = 0; j < DTW; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) vf[j][h] = buffer_load16(v, v_at + (j * 2 + h) * 1024);
  };
  auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };      // (loads stay on their way)

  f32x4 acc[DTW][RT];
#pragma unroll
  for (int j = 0; j < DTW; ++j)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[RT], l[RT];                             // what a row's weights refer to; the sum of this lane's weights
#pragma unroll
  for (int t = 0; t < RT; ++t) m[t] = -INFINITY, l[t] = 0.f;

  load_keys(pages[p_lo]);
  __syncthreads();
  for (int p = p_lo; p <= p_hi; ++p) {
    load_values(pages[p]);
    f32x4 s[RT];
    // (the fragments in LDS are read two k-steps ahead, and no earlier: there are no registers for more)
    bf16x8 ql[2][RT];
    auto from_lds = [&](int ks) {
#pragma unroll
      for (int t = 0; t < RT; ++t) ql[ks % 2][t] = *(const bf16x8*)&q_lds[ks][t][lane][0];
    };
#pragma unroll
    for (int ks = 0; ks < QS; ++ks) {
      if (ks >= QR - 2 && ks - QR + 2 < 2 && ks - QR + 2 < QL) from_lds(ks - QR + 2);
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const bf16x8 qa = qf[ks < QR ? ks : 0][t], qv = ql[ks % 2 ^ QR % 2][t];
        if (ks == 0) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(s[t]) : "a"(kf[ks]), "a"(qa));
        else if (ks < QR) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(s[t]) : "a"(kf[ks]), "a"(qa));
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(s[t]) : "a"(kf[ks]), "v"(qv));
      }
      if (ks >= QR && ks - QR + 2 < QL) from_lds(ks - QR + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    load_keys(pages[min(p + 1, p_hi)]);
    asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < RT; ++t) asm volatile("" : "+v"(s[t]));
    // s[t][e]: key p * 64 + wave * 16 + 4 g + e against row first + 16 t + i, times log2 e
#pragma unroll
    for (int t = 0; t < RT; ++t) s[t] *= scale;
    if (p * SYN_PAGE + SYN_PAGE - 1 > seen_by_all || p * SYN_PAGE <= unseen_by_some) {
      const int key0 = p * SYN_PAGE + wave * 16 + 4 * g;
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t][e] = (key0 + e <= pos[t]) & (key0 + e > unseen[t]) ? s[t][e] : -INFINITY;
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const float top = across16(fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3])), [](float x, float y) { return fmaxf(x, y); });
      if (g == 0) max_lds[t * 16 + i][wave] = top;
    }
    meet();                                       // (and everybody has done with the weights of the page before)
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const f32x4 tops = *(const f32x4*)&max_lds[t * 16 + i][0];
      const float top = fmaxf(fmaxf(tops[0], tops[1]), fmaxf(tops[2], tops[3]));
      const bool grown = top > m[t] + LA_LAZY || (m[t] == -INFINITY && top > m[t]);
      if (__any(grown)) {
        const float m_new = grown ? top : m[t];
        const float alpha = m[t] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[t] - m_new);
        m[t] = m_new, l[t] *= alpha;
#pragma unroll
        for (int j = 0; j < DTW; ++j) acc[j][t] *= alpha;
      }
      const float base = m[t] == -INFINITY ? 0.f : m[t];          // (a row that has seen nothing yet)
      bf16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float w = __builtin_amdgcn_exp2f(s[t][e] - base);
        l[t] += w;
        hi[e] = (bf16)w;
        lo[e] = (bf16)(w - (float)hi[e]);
      }
      *(bf16x4*)&p_lds[0][wave >> 1][t][lane][4 * (wave & 1)] = hi;
      *(bf16x4*)&p_lds[1][wave >> 1][t][lane][4 * (wave & 1)] = lo;
    }
    meet();
    // slots behind the sequence's end may hold anything: their weights are 0, their values are made 0 as well
    const int left = kv_len - p * SYN_PAGE;
    if (left < SYN_PAGE)
#pragma unroll
      for (int j = 0; j < DTW; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (32 * h + 4 * g + e >= left) vf[j][h][e] = (bf16)0.f;
            if (32 * h + 16 + 4 * g + e >= left) vf[j][h][4 + e] = (bf16)0.f;
          }
    asm volatile("s_nop 3" ::: "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 w[2][RT];
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int t = 0; t < RT; ++t) w[part][t] = *(const bf16x8*)&p_lds[part][h][t][lane][0];
#pragma unroll
      for (int part = 0; part < 2; ++part) {
#pragma unroll
        for (int j = 0; j < DTW; ++j)
#pragma unroll
          for (int t = 0; t < RT; ++t)
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[j][t]) : "v"(vf[j][h]), "v"(w[part][t]));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  // the sums of a row's weights: over the lanes, then over the waves
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    l[t] = across16(l[t], [](float x, float y) { return x + y; });
    if (g == 0) max_lds[t * 16 + i][wave] = l[t];      // (last read before the loop's last barrier)
  }
  meet();
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const f32x4 sums = *(const f32x4*)&max_lds[t * 16 + i][0];
    const float sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    const int flat = first + t * 16 + i;
    const float inv = 1.f / sum;
    if (flat > last) continue;
    // acc[j][t][e]: value (wave * DTW + j) * 16 + 4 g + e of the row
    bf16* orow = out + (row0 + flat) * rank + 4 * g;
#pragma unroll
    for (int j = 0; j < DTW; ++j)
      if (wave * DTW + j < n_dt) {
        bf16x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = (bf16)(acc[j][t][e] * inv);
        *(bf16x4*)(orow + (wave * DTW + j) * 16) = r;
      }
  }
}

// the splits of a tile merged in their order: the largest maximum, every split's sum and values scaled to it.
// One workgroup a (tile, row): the splits' maxima and sums fetched side by side, their factors in LDS, then a thread a
// value.
#define LA_MAX_SPLITS 1024
__global__ void __launch_bounds__(256)
latent_attention_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                              const int* __restrict__ seq_start, int n_seqs, bf16* __restrict__ out, int nh, int rank,
                              int n_splits) {
  __shared__ float factor[LA_MAX_SPLITS];
  __shared__ float red[16];
  const int gt = blockIdx.x, r = blockIdx.y;
  int seq, tile, start, rows;
  if (!la_find_unit(gt, LA_ROWS, seq_start, n_seqs, nh, seq, tile, start, rows)) return;
  const int flat = tile * LA_ROWS + r;
  if (flat >= rows) return;                 // (the whole workgroup)
  const size_t at0 = (size_t)gt * n_splits * LA_ROWS + r;
  float top = -INFINITY;
  for (int s = threadIdx.x; s < n_splits; s += blockDim.x) {
    const float ms = part_ml[2 * (at0 + (size_t)s * LA_ROWS)];
    factor[s] = ms;
    top = fmaxf(top, ms);
  }
  // the largest maximum of all splits: through LDS (block_sum's barriers also publish `factor`)
  top = wave_max(top);
  if (threadIdx.x % SYN_WAVE == 0) red[threadIdx.x / SYN_WAVE] = top;
  __syncthreads();
  float mm = -INFINITY;
  for (int w = 0; w < 4; ++w) mm = fmaxf(mm, red[w]);
  __syncthreads();
  float part = 0.f;
  for (int s = threadIdx.x; s < n_splits; s += blockDim.x) {
    const float ms = factor[s];
    const float f = ms == -INFINITY ? 0.f : expf(ms - mm);
    factor[s] = f;
    part += f * part_ml[2 * (at0 + (size_t)s * LA_ROWS) + 1];
  }
  const float l = block_sum(part, red);
  bf16* orow = out + ((size_t)(start + flat / nh) * nh + flat % nh) * rank;
  for (int d = threadIdx.x; d < rank; d += blockDim.x) {
    float o = 0.f;
    // eight splits' values on their way together, added in their order (8 rows of 32 heads, 42 splits: 12.2 ->
    // 6.8 us); a split without keys
    // weighs nothing and may hold anything
    for (int s0 = 0; s0 < n_splits; s0 += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part_o[(at0 + (size_t)min(s0 + u, n_splits - 1) * LA_ROWS) * rank + d];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float f = s0 + u < n_splits ? factor[s0 + u] : 0.f;
        if (f != 0.f) o += f * v[u];
      }
    }
    orow[d] = (bf16)(o / l);
  }
}

// share: a tile a workgroup (few tiles: single tokens), else four of a sequence and no splits.  n_tiles: the workgroups, at least the number of all sequences' tiles (share) or groups of four tiles;
// with share at least the number of tiles of all sequences, sum_b ceil(new tokens_b * heads / 16) (the host may not know
// the counts: (n_tokens * heads + 15) / 16 + n_seqs bounds it).  workspace: floats for n_tiles * n_splits * 16 *
// (rank + 2), used when n_splits > 1.
SYN_EXPORT int syn_latent_attention_bf16(const void* q, const void* k_pages, const void* v_pages, const int* page_table,
                                         int table_stride, const int* seq_start, const int* seq_past, int n_seqs,
                                         void* out, float* workspace, long workspace_floats, float scale, int n_tiles,
                                         int nh, int rank, int rot, int window, int n_splits, int share,
                                         hipStream_t stream) {
  const int R = rank + rot;
  SYN_CHECK(n_seqs > 0 && n_tiles > 0 && nh > 0, "latent_attention: empty input");
  SYN_CHECK(rank > 0 && rank % 16 == 0 && rank <= 512 && R % 16 == 0 && R <= 640,
            "latent_attention: rows of %d + %d values (multiples of 16 up to 512 and 640 together)", rank, rot);
  SYN_CHECK(window >= 0 && n_splits >= 1 && n_splits <= LA_MAX_SPLITS, "latent_attention: window %d, %d splits", window, n_splits);
  SYN_CHECK(n_splits == 1 || (workspace != nullptr && workspace_floats >= (long)n_tiles * n_splits * LA_ROWS * (rank + 2)),
            "latent_attention: a workspace of %ld floats for %d tiles in %d splits", workspace_floats, n_tiles, n_splits);
  SYN_CHECK(share || n_splits == 1, "latent_attention: pages are cut into splits only where a workgroup shares a tile");
  float* part_o = workspace;
  float* part_ml = workspace ? workspace + (size_t)n_tiles * n_splits * LA_ROWS * rank : nullptr;
  const bool x32 = R % 32 == 0;
#define SYN_LA_TILES(DT, QS, X)                                                                                             \
  latent_attention_bf16_kernel<DT, QS, X><<<dim3(share ? n_tiles : 4 * n_tiles, n_splits), 256, 0, stream>>>(               \
      (const bf16*)q, (const bf16*)k_pages, (const bf16*)v_pages, page_table, table_stride, seq_start, seq_past, n_seqs, \
      (bf16*)out, part_o, part_ml, scale, nh, rank, R, window, n_splits)
#define SYN_LA_PROMPT(DTW, QS, WHOLE)                                                                                    \
  latent_prompt_bf16_kernel<DTW, QS, WHOLE><<<n_tiles, 256, 0, stream>>>(                                                \
      (const bf16*)q, (const bf16*)k_pages, (const bf16*)v_pages, page_table, table_stride, seq_start, seq_past, n_seqs, \
      (bf16*)out, scale, nh, rank, R, window)
  // (rows of the queries that are no multiples of 32 were never asked to start at 16 bytes)
  const bool chunks = ((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0;
  if (!share && (x32 || chunks)) {
    if (rank <= 128 && R <= 160) SYN_LA_PROMPT(2, 5, false);
    else if (rank <= 256 && R <= 320) SYN_LA_PROMPT(4, 10, false);
    else if (R == 576) SYN_LA_PROMPT(8, 18, true);
    else SYN_LA_PROMPT(8, 20, false);
  } else if (rank <= 128 && R <= 160) {
    if (x32) SYN_LA_TILES(8, 5, true); else SYN_LA_TILES(8, 10, false);
  } else if (rank <= 256 && R <= 320) {
    if (x32) SYN_LA_TILES(16, 10, true); else SYN_LA_TILES(16, 20, false);
  } else {
    if (x32) SYN_LA_TILES(32, 20, true); else SYN_LA_TILES(32, 40, false);
  }
#undef SYN_LA_TILES
#undef SYN_LA_PROMPT
  SYN_LAUNCH_CHECK("latent_attention");
  if (n_splits > 1) {
    latent_attention_merge_kernel<<<dim3((n_tiles + 3) / 4 * 4, LA_ROWS), 256, 0, stream>>>(part_o, part_ml, seq_start, n_seqs,
                                                                                            (bf16*)out, nh, rank, n_splits);
    SYN_LAUNCH_CHECK("latent_attention_merge");
  }
  return 0;
}

// ------------------------------------------------------------------ prompts over keys and values of the heads' own
// The products with W_uk and W_uv at the keys' side after all: keys and values of every head are made from the latents once a step
// (two products over the sequences' rows), and a query then meets dim + rot instead of rank + rot values and sums v_dim instead
// of rank: with heads of 128 + 64 and a latent of 512 a (query, key) pair is 640 + 256 multiplications less 2,176 + 1,024 (the second
// numbers: a weight counts as two bf16 numbers, as above), which pays where a step brings as many tokens as a prompt.
//   latent_rows      the rows [latent | rotated part] of all sequences out of their pages, one after another, each sequence's first
//                    visible page first; what lies behind a sequence's end is zero
//   latent_expanded  the attention itself: 128 queries of a head a workgroup, four waves of 32, 32x32x16 matrix instructions,
//                    blocks of 64 keys through two LDS buffers, as csrc/attention_bf16.hip has them for 128 + 128
// Two workgroups a compute unit (80 KB of LDS each).  1,500 tokens, 32 heads of 128 + 64, a latent of 512: 61 + 220 + 55 us a
// layer with the up-projections absorbed (queries, attention, values), 5 + 37 + 73 so (rows, keys and values, attention).
#define LX_ROWS 128
#define LX_DIM 128           // of a head's unrotated keys and of its values
#define LX_ROT 64
#define LX_LAZY 8.f          // a row's sums are rescaled where its maximum has grown by more than 2^LX_LAZY

// rows of the sequences in front of `seq`, and the first page of `seq` that some new token sees
__device__ __forceinline__ int lx_rows_before(const int* seq_start, const int* seq_past, int seq, int window, int& first_page) {
  const int lane = threadIdx.x % SYN_WAVE;
  int pages = 0;
  for (int b = lane; b < seq; b += SYN_WAVE) {
    const int past = seq_past[b], len = past + seq_start[b + 1] - seq_start[b];
    pages += (len + SYN_PAGE - 1) / SYN_PAGE - (window > 0 ? max(0, past - window + 1) / SYN_PAGE : 0);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) pages += __shfl_xor(pages, off, SYN_WAVE);
  first_page = (window > 0 ? max(0, seq_past[seq] - window + 1) : 0) / SYN_PAGE;
  return pages * SYN_PAGE;
}

__global__ void __launch_bounds__(256)
latent_rows_kernel(const bf16* __restrict__ k_pages, const int* __restrict__ page_table, int table_stride,
                   const int* __restrict__ seq_start, const int* __restrict__ seq_past, int n_seqs, int window, int rank, int rot,
                   bf16* __restrict__ latent, bf16* __restrict__ rotated) {
  // a quarter of a page a workgroup; which page this is: the sequences one after another
  int t = blockIdx.x / 4, seq = 0, page = 0, len = 0;
  for (; seq < n_seqs; ++seq) {
    const int past = seq_past[seq];
    len = past + seq_start[seq + 1] - seq_start[seq];
    const int lo = (window > 0 ? max(0, past - window + 1) : 0) / SYN_PAGE, n = (len + SYN_PAGE - 1) / SYN_PAGE - lo;
    if (t < n) {
      page = lo + t;
      break;
    }
    t -= n;
  }
  if (seq == n_seqs) return;
  const int R = rank + rot, per = R / 8, left = len - page * SYN_PAGE;
  const bf16* src = k_pages + (size_t)page_table[(size_t)seq * table_stride + page] * SYN_PAGE * R;
  const bf16x8 zero = {};
  for (int c = threadIdx.x; c < SYN_PAGE / 4 * per; c += blockDim.x) {
    const int r = blockIdx.x % 4 * (SYN_PAGE / 4) + c / per, d = c % per * 8;
    const bf16x8 v = r < left ? *(const bf16x8*)(src + (size_t)r * R + d) : zero;
    const size_t row = (size_t)(blockIdx.x / 4) * SYN_PAGE + r;
    *(bf16x8*)(d < rank ? latent + row * rank + d : rotated + row * rot + d - rank) = v;
  }
}

__global__ void __launch_bounds__(256, 2)
latent_expanded_kernel(const bf16* __restrict__ q_nope, const bf16* __restrict__ q_rot, int q_rot_stride, const bf16* __restrict__ keys,
                       const bf16* __restrict__ rotated, const bf16* __restrict__ values, int n_rows,
                       const int* __restrict__ seq_start, const int* __restrict__ seq_past, int n_seqs, bf16* __restrict__ out,
                       float scale, int nh, int first_head, int all_heads, int window, const float* __restrict__ gate, int gate_stride,
                       int gate_per_value) {
  constexpr int KS = (LX_DIM + LX_ROT) / 16, NOPE = SYN_PAGE * LX_DIM * 2, ROT = SYN_PAGE * LX_ROT * 2, BUF = 2 * NOPE + ROT;
  constexpr int DT = LX_DIM / 16, D32 = LX_DIM / 32, NLOAD = BUF / 1024 / 4, AHEAD = 6;
  extern __shared__ __attribute__((aligned(16))) char lds[];      // [2][unrotated keys | rotated keys | values]
  // late tiles of a sequence see the most keys: they come first, and a late and an early one meet on a compute unit
  int total = 0;
  for (int s = 0; s < n_seqs; ++s) total += (seq_start[s + 1] - seq_start[s] + LX_ROWS - 1) / LX_ROWS;
  const int y = blockIdx.y, half = (total + 1) / 2;
  if (y >= total) return;
  int seq, tile, tok0, n_new;
  if (!la_find_unit(y < half ? total - 1 - y : y - half, LX_ROWS, seq_start, n_seqs, 1, seq, tile, tok0, n_new)) return;
  seq = __builtin_amdgcn_readfirstlane(seq), tile = __builtin_amdgcn_readfirstlane(tile);
  tok0 = __builtin_amdgcn_readfirstlane(tok0), n_new = __builtin_amdgcn_readfirstlane(n_new);
  const int lane = threadIdx.x % SYN_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SYN_WAVE);
  const int n32 = lane % 32, hh = lane / 32;
  const int hx = blockIdx.x, head = nh % 8 == 0 ? (hx % 8) * (nh / 8) + hx / 8 : hx;      // neighbouring heads on one die
  const int past = seq_past[seq], q0 = tile * LX_ROWS;
  int page0;
  const int row0 = __builtin_amdgcn_readfirstlane(lx_rows_before(seq_start, seq_past, seq, window, page0));
  const int kb_hi = (past + min(q0 + LX_ROWS, n_new) - 1) / SYN_PAGE;
  const int kb_lo = (window > 0 ? max(0, past + q0 - window + 1) : 0) / SYN_PAGE;
  if (row0 + (kb_hi - page0 + 1) * SYN_PAGE > n_rows) return;      // (the caller's rows are not those of these sequences)
  const int r0 = q0 + wave * 32, row = r0 + n32;
  const bool wave_on = r0 < n_new, valid = row < n_new;
  const int qpos = valid ? past + row : -1, lo = (window > 0 && valid) ? max(0, qpos - window + 1) : 0;
  const int w_kmax = past + min(r0 + 31, n_new - 1), w_qmin = past + r0, w_kmin = window > 0 ? max(0, w_qmin - window + 1) : 0;
  const float scale2 = scale * 1.4426950408889634f;
  const bf16x8 zero8 = {};
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d = 16 * ks + 8 * hh;
    const size_t at = (size_t)(tok0 + row) * all_heads + first_head + head;
    qf[ks] = !valid ? zero8 : ks < LX_DIM / 16 ? *(const bf16x8*)(q_nope + at * LX_DIM + d) : *(const bf16x8*)(q_rot + at * q_rot_stride + d - LX_DIM);
  }
  f32x16 o[D32];
#pragma unroll
  for (int d = 0; d < D32; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  struct Views {
    BufferView k, r, v;
  };
  auto views_of = [&](int kb) {
    const size_t at = row0 + (size_t)(kb - page0) * SYN_PAGE;
    return Views{buffer_view(keys + (at * nh + head) * LX_DIM, ((size_t)(SYN_PAGE - 1) * nh + 1) * LX_DIM * 2),
                 buffer_view(rotated + at * LX_ROT, ROT),
                 buffer_view(values + (size_t)head * LX_DIM * n_rows + at, ((size_t)(LX_DIM - 1) * n_rows + SYN_PAGE) * 2)};
  };
  // load j of a wave for a block: 1 KB straight into LDS, 16-byte chunks of a key's row swizzled (a fragment reads 32 rows at the same
  // column), values in the order of their fragments
  auto fetch_one = [&](const Views& v, int buf, int j) {
    char* dst = lds + buf * BUF;
    const int i = j * 4 + wave;
    if (j < 4) {
      const int at = 64 * i + lane, r = at / 16, slot = at % 16;
      buffer_to_lds16(v.k, dst + 1024 * i, (unsigned)(r * nh * LX_DIM * 2 + (slot ^ (r & 15)) * 16), 0);
    } else if (j < 6) {
      const int at = 64 * (i - 16) + lane, r = at / 8, slot = at % 8;
      buffer_to_lds16(v.r, dst + 1024 * i, (unsigned)((r * 8 + (slot ^ ((r >> 1) & 7))) * 16), 0);
    } else {
      const int f = i - 24, d = (f % DT) * 16 + lane % 16, key = (f / DT) * 32 + (lane / 16) * 8;
      buffer_to_lds16(v.v, dst + 1024 * i, (unsigned)((d * n_rows + key) * 2), 0);
    }
  };
  auto landed = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's loads have written LDS; behind the barrier all have
    __syncthreads();
  };
  const int krow0 = 16 * (n32 / 16) + 8 * ((n32 % 8) / 4) + 4 * ((n32 % 16) / 8) + n32 % 4;      // (so that a lane's scores are 8 consecutive keys)

  auto block = [&](int kb, auto more) {
    constexpr bool MORE = decltype(more)::value;
    const int buf = (kb - kb_lo) & 1, key0 = kb * SYN_PAGE;
    Views next;
    if constexpr (MORE) next = views_of(kb + 1);
    const char* ks_ = lds + buf * BUF;
    const char* rs_ = ks_ + NOPE;
    const char* vs_ = rs_ + ROT;
    if (wave_on && key0 <= w_kmax && key0 + SYN_PAGE > w_kmin) {
      constexpr int NQK = 2 * KS, NPV = 4 * D32;
      static_assert(NLOAD <= NQK / 2, "a load behind every second MFMA of the scores");
      f32x16 s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t][e] = 0.f;
      auto k_frag = [&](int i) {   // read i: k-step i / 2 of score tile i % 2
        const int ks = i / 2, r = 32 * (i % 2) + krow0;
        return ks < LX_DIM / 16 ? *(const bf16x8*)(ks_ + (r * 16 + ((2 * ks + hh) ^ (r & 15))) * 16)
                                : *(const bf16x8*)(rs_ + (r * 8 + ((2 * (ks - LX_DIM / 16) + hh) ^ ((r >> 1) & 7))) * 16);
      };
      auto v_frag = [&](int i) {   // read i: output tile i % D32 of k-step i / D32 = 2 t + j
        const int d = i % D32, tj = i / D32, t = tj / 2, j = tj % 2;
        return *(const bf16x8*)(vs_ + (((t * DT + 2 * d + n32 / 16) * 64 + (2 * j + hh) * 16 + n32 % 16)) * 16);
      };
      bf16x8 kf[NQK], vf[NPV];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) kf[i] = k_frag(i);
#pragma unroll
      for (int i = 0; i < NQK; ++i) {
        s[i % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[i], qf[i / 2], s[i % 2], 0, 0, 0);
        if (i + AHEAD < NQK) kf[i + AHEAD] = k_frag(i + AHEAD);
        else if (i + AHEAD - NQK < AHEAD) vf[i + AHEAD - NQK] = v_frag(i + AHEAD - NQK);
        if (MORE && i % 2 == 1 && i / 2 < NLOAD) fetch_one(next, buf ^ 1, i / 2);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
      for (int i = 0; i < NQK; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA,
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one read behind it,
        if (MORE && i % 2 == 1 && i / 2 < NLOAD) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);      // a load behind every second
      }
      __builtin_amdgcn_sched_barrier(0);
      if (key0 + SYN_PAGE - 1 > w_qmin || (window > 0 && key0 < w_kmax - window + 1) || r0 + 32 > n_new) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int key = key0 + 32 * t + 16 * (e / 8) + 8 * hh + e % 8;
            if (key > qpos || key < lo) s[t][e] = -INFINITY;
          }
      }
      float mloc = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mloc = fmaxf(mloc, s[t][e]);
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32, SYN_WAVE)) * scale2;
      const bool raise = mloc > m_run + LX_LAZY || (m_run == -INFINITY && mloc > -INFINITY);
      if (__any(raise)) {
        const float m_new = raise ? mloc : m_run;
        const float alpha = raise ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;  // from -inf: 0
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < D32; ++d) o[d] *= alpha;
      }
      const float neg_m = m_run == -INFINITY ? 0.f : -m_run;  // a column that has seen no key yet
      float lsum = 0.f;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int tj = 0; tj < 4; ++tj) {
        bf16x8 hi, rest;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[tj / 2][8 * (tj % 2) + e], scale2, neg_m));   // a masked score: 2^-inf = 0
          lsum += p;
          hi[e] = (bf16)p;
          rest[e] = (bf16)(p - (float)hi[e]);
        }
#pragma unroll
        for (int d = 0; d < D32; ++d) {
          const int i = tj * D32 + d;
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], hi, o[d], 0, 0, 0);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], rest, o[d], 0, 0, 0);
          if (i + AHEAD < NPV) vf[i + AHEAD] = v_frag(i + AHEAD);
        }
      }
      l_run += lsum;
    } else if constexpr (MORE) {
#pragma unroll
      for (int j = 0; j < NLOAD; ++j) fetch_one(next, buf ^ 1, j);
    }
    landed();
  };
  {
    const Views v = views_of(kb_lo);
#pragma unroll
    for (int j = 0; j < NLOAD; ++j) fetch_one(v, 0, j);
  }
  landed();
  for (int kb = kb_lo; kb < kb_hi; ++kb) block(kb, std::true_type{});
  block(kb_hi, std::false_type{});
  if (!wave_on) return;
  const float l = l_run + __shfl_xor(l_run, 32, SYN_WAVE);
  if (!valid) return;
  const float inv = 1.f / l;
  const size_t at = (size_t)(tok0 + row) * all_heads + first_head + head;
  const float* grow = gate ? gate + (size_t)(tok0 + row) * gate_stride + (first_head + head) * (gate_per_value ? LX_DIM : 1) : nullptr;
  auto sigmoid = [](float z) { return 1.f / (1.f + expf(-z)); };
  const float of_head = gate && !gate_per_value ? sigmoid(grow[0]) : 1.f;
  bf16* orow = out + at * LX_DIM + 4 * hh;
#pragma unroll
  for (int d = 0; d < D32; ++d)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = o[d][4 * b + e] * inv;
        if (gate) x *= gate_per_value ? sigmoid(grow[32 * d + 8 * b + 4 * hh + e]) : of_head;
        v[e] = (bf16)x;
      }
      *(bf16x4*)(orow + 32 * d + 8 * b) = v;
    }
}

// The rows of a step's sequences out of their pages: latent [n_rows][rank], rotated [n_rows][rot], n_rows = 64 times the pages that some
// new token of its sequence sees (window 0: all).
SYN_EXPORT int syn_latent_rows(const void* k_pages, const int* page_table, int table_stride, const int* seq_start, const int* seq_past,
                               int n_seqs, int window, int rank, int rot, void* latent, void* rotated, int n_rows, hipStream_t stream) {
  SYN_CHECK(n_seqs > 0 && n_rows > 0 && n_rows % SYN_PAGE == 0 && window >= 0, "latent_rows: %d rows of %d sequences", n_rows, n_seqs);
  SYN_CHECK(rank > 0 && rot >= 0 && rank % 8 == 0 && rot % 8 == 0 && ((uintptr_t)k_pages | (uintptr_t)latent | (uintptr_t)rotated) % 16 == 0,
            "latent_rows: rows of %d + %d values (multiples of 8, 16-byte aligned)", rank, rot);
  latent_rows_kernel<<<4 * (n_rows / SYN_PAGE), 256, 0, stream>>>((const bf16*)k_pages, page_table, table_stride, seq_start, seq_past, n_seqs,
                                                            window, rank, rot, (bf16*)latent, (bf16*)rotated);
  SYN_LAUNCH_CHECK("latent_rows");
  return 0;
}

// The nh heads from first_head on of all_heads: q_nope [N][all_heads][128]; q_rot: the rotated parts, 64 values every q_rot_stride; keys
// [n_rows][nh][128], rotated [n_rows][64], values [nh][128][n_rows] (rows as syn_latent_rows leaves them); out [N][all_heads][128] times
// sigmoid(gate), gate float rows every gate_stride: one number a head or (gate_per_value) a value, or null.
SYN_EXPORT int syn_latent_expanded(const void* q_nope, const void* q_rot, int q_rot_stride, const void* keys, const void* rotated,
                                   const void* values, int n_rows, const int* seq_start, const int* seq_past, int n_seqs, int n_tokens,
                                   void* out, float scale, int nh, int first_head, int all_heads, int dim, int rot, int window,
                                   const float* gate, int gate_stride, int gate_per_value, hipStream_t stream) {
  SYN_CHECK(dim == LX_DIM && rot == LX_ROT, "latent_expanded: heads of %d + %d values (%d + %d)", dim, rot, LX_DIM, LX_ROT);
  SYN_CHECK(n_seqs > 0 && n_tokens >= n_seqs && nh > 0 && n_rows > 0 && n_rows % SYN_PAGE == 0 && window >= 0 && scale > 0.f,
            "latent_expanded: %d tokens, %d rows, scale %g", n_tokens, n_rows, (double)scale);
  SYN_CHECK(first_head >= 0 && first_head + nh <= all_heads, "latent_expanded: heads %d to %d of %d", first_head, first_head + nh, all_heads);
  SYN_CHECK(q_rot_stride % 8 == 0 && ((uintptr_t)q_nope | (uintptr_t)q_rot | (uintptr_t)keys | (uintptr_t)rotated | (uintptr_t)values | (uintptr_t)out) % 16 == 0,
            "latent_expanded: operands must be 16-byte aligned");
  SYN_CHECK((size_t)n_rows * LX_DIM * 2 < 0x7fffffffull && (size_t)nh * LX_DIM * 2 * SYN_PAGE < 0x7fffffffull, "latent_expanded: %d rows of %d heads", n_rows, nh);
  constexpr int LDS = 2 * (2 * SYN_PAGE * LX_DIM + SYN_PAGE * LX_ROT) * 2;
  static OncePerDevice raised;
  const hipError_t e = once_per_device(raised, [&] {
    return hipFuncSetAttribute((const void*)latent_expanded_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  SYN_CHECK(e == hipSuccess, "latent_expanded: %d bytes of LDS refused: %s", LDS, hipGetErrorString(e));
  const int tiles = n_tokens / LX_ROWS + n_seqs;      // a bound; surplus workgroups leave at once
  SYN_CHECK(tiles <= 65535, "latent_expanded: %d tiles", tiles);
  latent_expanded_kernel<<<dim3(nh, tiles), 256, LDS, stream>>>((const bf16*)q_nope, (const bf16*)q_rot, q_rot_stride, (const bf16*)keys,
                                                                (const bf16*)rotated, (const bf16*)values, n_rows, seq_start, seq_past,
                                                                n_seqs, (bf16*)out, scale, nh, first_head, all_heads, window, gate, gate_stride,
                                                                gate_per_value);
  SYN_LAUNCH_CHECK("latent_expanded");
  return 0;
}
