// Products of rows with one of several weight matrices, chosen by the row's group:
//
//   out[orow(r), b, n] = epilogue( sum_k A[arow(r), b, k] * W[b, n, k] )         b: the group (an expert, a head)
//
// Two ways to say which rows meet which matrix:
//   * segments: seg_start[b] <= r < seg_start[b + 1] are the rows of group b (tokens sorted by expert), with
//     arow(r) = a_rows[r] and orow(r) = o_rows[r] gathered through index lists;
//   * every group takes all M rows (a linear map for each head of a token): A, W and out move on by a fixed
//     number of elements from one group to the next.
// Epilogue, in this order and each optional: the exact GELU 0.5 z (1 + erf(z / sqrt 2)) or max(z, 0)^2; a weight of the row;
// sigmoid of a gate value read from float rows.  Or, with `pair`: W's rows come in pairs (2 j: the gate row of output j,
// 2 j + 1: its up row) and what is stored is the gated activation of the two sums (gated, csrc/common.h), N / 2 columns.  Sums are 32-bit.  bf16 operands whose K is a multiple of 32 run on
// the matrix cores: with few rows a group 16x16x32 with operands straight from memory as 16-byte pieces of rows (no
// LDS: a wave computes 32 rows x 64 columns), with many rows tiles of 128 x 128 through LDS (any K that is a multiple
// of 8); everything else, and all of the 32-bit path, is plain FMA with one wave a (row, 8 columns).
//
// Beside it: the choice of a mixture's router (the largest `top` logits of a token, softmax over those) and the
// counting sort that turns the choices into segments.
#include <type_traits>

#include "common.h"

struct GroupedArgs {
  const void* a;
  long lda, a_group;        // A[row, group, k] = a[row * lda + group * a_group + k]
  const void* w;
  long w_group, ldw;        // W[group, n, k] = w[group * w_group + n * ldw + k]
  void* out;
  long ldo, o_group;        // out[row, group, n] = out[row * ldo + group * o_group + n]
  int out_is_f32;
  const int* seg_start;     // [groups + 1], or null: every group takes rows 0 .. M - 1
  const int* a_rows;        // [rows] or null
  const int* o_rows;        // [rows] or null
  const float* row_weight;  // [rows] or null
  const float* gate;        // or null: gate[row * gate_ld + group * gate_group + n * gate_col]
  long gate_ld, gate_group;
  int gate_col;
  int act;                  // 0: none, 1: exact GELU, 2: max(z, 0)^2
  int pair;                 // 0: none; else 1 + the code of the gated activation over pairs of rows of W
  float limit;              // that activation's bound, if it has one
  int M, N, K, groups;
  int w_packed;             // W[group] lies in the order of the fragments: [N / 16][K / 32][64 lanes][8] with
                            // lane = 16 (k % 32 / 8) + n % 16 (bf16, N a multiple of 16, K of 32); 0: plain rows
};

// element (n, k) of a matrix in fragment order, K32 = K / 32
__device__ __forceinline__ size_t packed_at(int n, int k, int K32) {
  return ((size_t)(n >> 4) * K32 + (k >> 5)) * 512 + (((k & 31) >> 3) << 7) + ((n & 15) << 3) + (k & 7);
}

__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }

__device__ __forceinline__ float grouped_epilogue(const GroupedArgs& g, float v, int r, int b, int n) {
  if (g.act == 1) v = gelu_erf(v);
  if (g.act == 2) v = point_activation(SYN_POINT_RELU_SQUARED, v);
  if (g.row_weight) v *= g.row_weight[r];
  if (g.gate) {
    const float z = g.gate[(size_t)r * g.gate_ld + (size_t)b * g.gate_group + (size_t)n * g.gate_col];
    v *= 1.f / (1.f + expf(-z));
  }
  return v;
}

// the pair (gate sum, up sum) of output column n / 2 (n even)
__device__ __forceinline__ float grouped_pair(const GroupedArgs& g, float gate, float up, int r) {
  float v = gated(g.pair - 1, gate, up, g.limit);
  if (g.row_weight) v *= g.row_weight[r];
  return v;
}

__device__ __forceinline__ void grouped_store(const GroupedArgs& g, int r, int b, int n, float v) {
  const int orow = g.o_rows ? g.o_rows[r] : r;
  const size_t at = (size_t)orow * g.ldo + (size_t)b * g.o_group + n;
  if (g.out_is_f32) ((float*)g.out)[at] = v;
  else ((bf16*)g.out)[at] = (bf16)v;
}

// ---------------------------------------------------------------- plain FMA: one wave a (row, 8 columns)
template <typename T>
__global__ void __launch_bounds__(256) grouped_product_simt_kernel(GroupedArgs g) {
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  int r = blockIdx.x, b = blockIdx.z;
  if (g.seg_start) {
    // the group whose segment holds row r (segments are in order and cover 0 .. seg_start[groups] - 1)
    if (r >= g.seg_start[g.groups]) return;
    int lo = 0, hi = g.groups;
    while (hi - lo > 1) {
      const int mid = (lo + hi) / 2;
      if (g.seg_start[mid] <= r) lo = mid; else hi = mid;
    }
    b = lo;
  }
  const int n0 = (blockIdx.y * 4 + wave) * 8;
  if (n0 >= g.N) return;
  const int arow = g.a_rows ? g.a_rows[r] : r;
  const T* a = (const T*)g.a + (size_t)arow * g.lda + (size_t)b * g.a_group;
  const T* w = (const T*)g.w + (size_t)b * g.w_group;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int k = lane; k < g.K; k += SYN_WAVE) {
    const float x = to_f32<T>(a[k]);
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (n0 + c < g.N)
        acc[c] = fmaf(x, to_f32<T>(w[g.w_packed ? packed_at(n0 + c, k, g.K / 32) : (size_t)(n0 + c) * g.ldw + k]), acc[c]);
  }
  if (g.pair) {
#pragma unroll
    for (int c = 0; c < 8; c += 2) {
      const float gate = wave_sum(acc[c]), up = wave_sum(acc[c + 1]);
      if (lane == 0 && n0 + c < g.N) grouped_store(g, r, b, (n0 + c) / 2, grouped_pair(g, gate, up, r));
    }
    return;
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float v = wave_sum(acc[c]);
    if (lane == 0 && n0 + c < g.N) grouped_store(g, r, b, n0 + c, grouped_epilogue(g, v, r, b, n0 + c));
  }
}

// ---------------------------------------------------------------- bf16 on the matrix cores
// D = W_tile (16 outputs x 32 k) . A_tile^T (32 k x 16 rows): a lane then holds four consecutive outputs of one row.
// Both operands are 16-byte pieces of rows (8 k-values of lane group lane / 16), so whatever order the instruction
// gives the k-values inside a lane group, the two operands agree.
#define GP_TM 32
// NB: blocks of 16 outputs a wave (4: 64 outputs; 1: 16 outputs, four times the waves, where few groups have rows and
// each group's matrix has to be streamed by more than a few waves).
template <int NB>
__global__ void __launch_bounds__(256) grouped_product_mfma_kernel(GroupedArgs g) {
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE, i = lane % 16, q = lane / 16;
  int b = blockIdx.z, row0, row_end;
  if (g.seg_start) {
    int t = blockIdx.x;
    b = -1;
    for (int e = 0; e < g.groups; ++e) {
      const int s0 = g.seg_start[e], n = g.seg_start[e + 1] - s0, tiles = (n + GP_TM - 1) / GP_TM;
      if (t < tiles) {
        b = e, row0 = s0 + t * GP_TM, row_end = s0 + n;
        break;
      }
      t -= tiles;
    }
    if (b < 0) return;
  } else {
    row0 = blockIdx.x * GP_TM, row_end = g.M;
    if (row0 >= row_end) return;
  }
  const int n0 = (blockIdx.y * 4 + wave) * 16 * NB;
  if (n0 >= g.N) return;
  const bf16* A = (const bf16*)g.a + (size_t)b * g.a_group;
  const bf16* W = (const bf16*)g.w + (size_t)b * g.w_group;
  // rows beyond the segment and outputs beyond N read row 0 (a valid address) and count as zeros
  const bf16* arow[2];
  bool a_ok[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int r = row0 + mb * 16 + i;
    a_ok[mb] = r < row_end;
    const int src = a_ok[mb] ? (g.a_rows ? g.a_rows[r] : r) : (g.a_rows ? g.a_rows[row0] : row0);
    arow[mb] = A + (size_t)src * g.lda + q * 8;
  }
  const bf16* wrow[NB];
  bool w_ok[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = n0 + nb * 16 + i;
    w_ok[nb] = n < g.N;
    // (in fragment order a wave's load of a k-step is 1 KB of consecutive bytes, and the next k-step lies 1 KB on)
    wrow[nb] = g.w_packed ? W + (size_t)((w_ok[nb] ? n : 0) >> 4) * (g.K / 32) * 512 + lane * 8
                          : W + (size_t)(w_ok[nb] ? n : 0) * g.ldw + q * 8;
  }
  const int w_step = g.w_packed ? 512 : 32;          // elements from one k-step of 32 to the next
  f32x4 acc[2][NB];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  // several k-steps at a time: their loads (24) are asked for together (a group's matrix is read once, as a stream), then
  // multiplied; the k-steps that are left over follow one by one
  constexpr int AHEAD = NB == 1 ? 8 : 4;
  int k0 = 0;
  for (; k0 + 32 * AHEAD <= g.K; k0 += 32 * AHEAD) {
    bf16x8 xa[AHEAD][2], xw[AHEAD][NB];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) xa[u][mb] = *(const bf16x8*)(arow[mb] + k0 + 32 * u);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) xw[u][nb] = __builtin_nontemporal_load((const bf16x8*)(wrow[nb] + (size_t)(k0 / 32 + u) * w_step));
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) xa[u][mb] = a_ok[mb] ? xa[u][mb] : zero;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) xw[u][nb] = w_ok[nb] ? xw[u][nb] : zero;
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xw[u][nb], xa[u][mb], acc[mb][nb], 0, 0, 0);
    }
  }
  for (; k0 < g.K; k0 += 32) {
    bf16x8 xa[2], xw[NB];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) xa[mb] = a_ok[mb] ? *(const bf16x8*)(arow[mb] + k0) : zero;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) xw[nb] = w_ok[nb] ? *(const bf16x8*)(wrow[nb] + (size_t)(k0 / 32) * w_step) : zero;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xw[nb], xa[mb], acc[mb][nb], 0, 0, 0);
  }
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int r = row0 + mb * 16 + i;
    if (r >= row_end) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + nb * 16 + q * 4 + e;
        if (g.pair) {      // (a lane holds four consecutive outputs: two pairs)
          if (e % 2 == 0 && n < g.N) grouped_store(g, r, b, n / 2, grouped_pair(g, acc[mb][nb][e], acc[mb][nb][e + (e % 2 == 0)], r));
        } else if (n < g.N) {
          grouped_store(g, r, b, n, grouped_epilogue(g, acc[mb][nb][e], r, b, n));
        }
      }
  }
}

// ---------------------------------------------------------------- bf16 on the matrix cores, many rows a group
// Tiles of 128 rows x 128 outputs x 64 k through LDS (double-buffered: while one k-tile is multiplied the next is on
// its way from memory into registers), four waves of 64 x 64 each, MFMA 32x32x16: A = rows of x, B = rows of W,
// D[m = 8 (e / 4) + 4 (lane / 32) + e % 4][n = lane % 32].  Rows of x are gathered through a_rows on their way into
// LDS.  K is a multiple of 8 (a 16-byte chunk lies inside or outside as a whole).
#define GT_BM 128
#define GT_BN 128
#define GT_BK 64
#define GT_LD (GT_BK + 8)
template <bool PAIR>
__global__ void __launch_bounds__(256) grouped_product_tiled_kernel(GroupedArgs g) {
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];      // [2][(GT_BM + GT_BN) * GT_LD]
  const int tid = threadIdx.x, wave = tid / SYN_WAVE, lane = tid % SYN_WAVE;
  // Workgroups go to the eight XCDs in turns, each with an L2 of its own: workgroup w takes place
  // (w % 8) * (places / 8) + w / 8 of the order (row tile, column tile), so that one XCD walks the column tiles of a
  // few row tiles: it reads those rows of x once, and a group's matrix for the group's few row tiles in a row.
  const int col_tiles = (g.N + GT_BN - 1) / GT_BN;
  const int places = gridDim.x;                       // a multiple of 8
  const int place = (blockIdx.x % 8) * (places / 8) + blockIdx.x / 8;
  int b = blockIdx.z, row0, row_end;
  if (g.seg_start) {
    int t = place / col_tiles;
    b = -1;
    for (int e = 0; e < g.groups; ++e) {
      const int s0 = g.seg_start[e], n = g.seg_start[e + 1] - s0, tiles = (n + GT_BM - 1) / GT_BM;
      if (t < tiles) {
        b = e, row0 = s0 + t * GT_BM, row_end = s0 + n;
        break;
      }
      t -= tiles;
    }
    if (b < 0) return;                      // (the whole workgroup, before any barrier)
  } else {
    row0 = (place / col_tiles) * GT_BM, row_end = g.M;
    if (row0 >= row_end) return;
  }
  const int n0 = (place % col_tiles) * GT_BN;
  const int wm = (wave / 2) * 64, wn = (wave % 2) * 64;
  constexpr int CPR = GT_BK / 8, RPP = 256 / CPR, XL = GT_BM / RPP, WL = GT_BN / RPP;
  const int lrow = tid / CPR, lchunk = (tid % CPR) * 8;
  const bf16* A = (const bf16*)g.a + (size_t)b * g.a_group;
  const bf16* W = (const bf16*)g.w + (size_t)b * g.w_group;
  const bf16* xg[XL];
  const bf16* wg[WL];
  bool xin[XL], win[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int r = row0 + lrow + RPP * i;
    xin[i] = r < row_end;
    const int src = xin[i] ? (g.a_rows ? g.a_rows[r] : r) : 0;
    xg[i] = A + (size_t)src * g.lda + lchunk;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int n = n0 + lrow + RPP * i;
    win[i] = n < g.N;
    const int nn = win[i] ? n : 0;
    wg[i] = g.w_packed ? W + (size_t)(nn >> 4) * (g.K / 32) * 512 + ((nn & 15) << 3) + ((lchunk >> 5) << 9) + (((lchunk & 31) >> 3) << 7)
                       : W + (size_t)nn * g.ldw + lchunk;
  }
  const int w_tile = g.w_packed ? (GT_BK / 32) * 512 : GT_BK;      // elements from one k-tile to the next
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const int nk = (g.K + GT_BK - 1) / GT_BK;
  bf16x8 rx[XL], rw[WL];
  auto fetch = [&](int kt) {
    const int k = kt * GT_BK;
    const bool kin = k + lchunk < g.K;
#pragma unroll
    for (int i = 0; i < XL; ++i) rx[i] = (kin && xin[i]) ? *(const bf16x8*)(xg[i] + k) : zero;
#pragma unroll
    for (int i = 0; i < WL; ++i) rw[i] = (kin && win[i]) ? *(const bf16x8*)(wg[i] + (size_t)kt * w_tile) : zero;
  };
  auto stash = [&](int buf) {
    bf16* xs = smem + buf * (GT_BM + GT_BN) * GT_LD;
    bf16* ws = xs + GT_BM * GT_LD;
#pragma unroll
    for (int i = 0; i < XL; ++i) *(bf16x8*)(xs + (lrow + RPP * i) * GT_LD + lchunk) = rx[i];
#pragma unroll
    for (int i = 0; i < WL; ++i) *(bf16x8*)(ws + (lrow + RPP * i) * GT_LD + lchunk) = rw[i];
  };
  fetch(0);
  stash(0);
  __syncthreads();
  const int fr = lane % 32, fk = (lane / 32) * 8;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) fetch(kt + 1);
    const bf16* xs = smem + buf * (GT_BM + GT_BN) * GT_LD;
    const bf16* ws = xs + GT_BM * GT_LD;
#pragma unroll
    for (int ks = 0; ks < GT_BK; ks += 16) {
      bf16x8 fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = *(const bf16x8*)(xs + (wm + i * 32 + fr) * GT_LD + ks + fk);
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = *(const bf16x8*)(ws + (wn + j * 32 + fr) * GT_LD + ks + fk);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) stash(buf ^ 1);      // the other buffer was last read before the previous barrier
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = row0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
        const int n = n0 + wn + j * 32 + lane % 32;
        if constexpr (PAIR) {      // (neighbouring lanes hold neighbouring outputs: the even lane takes its neighbour's up sum)
          const float up = __shfl_xor(acc[i][j][e], 1, SYN_WAVE);
          if (lane % 2 == 0 && r < row_end && n < g.N) grouped_store(g, r, b, n / 2, grouped_pair(g, acc[i][j][e], up, r));
        } else if (r < row_end && n < g.N) {
          grouped_store(g, r, b, n, grouped_epilogue(g, acc[i][j][e], r, b, n));
        }
      }
}

// ---------------------------------------------------------------- bf16, many rows a group, W in fragment order: streamed
// The scheme of the products of many rows (gemm_stream_kernel in gemm.hip: four waves with a quarter of the tile each,
// accumulators in place, k-tiles in rings of LDS buffers, x in whole lines of 128 bytes of a row, one stream of k-steps over all
// tiles of a workgroup) for rows sorted into segments: which tiles there are stands in seg_start, on the device, so every wave counts
// the segments' tiles into registers first and looks its tiles up there.  Rows of x are gathered by their loads (each lane asks for a
// piece of its own row), rows of the output and their weights looked up for the stores.
// What bounds it: what a compute unit takes in, since all of W comes from memory and x from L2 (a k-step of 256 x 256 takes 0.55 to 0.7
// us for 0.43 of MFMAs, with zeros as operands too), and the stores of a tile, which the next tile's first loads wait behind.  So
//   * a segment's tiles get the same number of rows, and a k-step leaves out the 32 rows at a time that a tile does not have;
//   * what the stores look up, and the next tile's row list, are asked for before the first store: behind stores they would wait
//     for these, once for every 32 rows;
//   * a last round of tiles for up to half of the workgroups is cut into halves of tiles for all.
// ONCE: W's loads are marked non-temporal, where a tile of W meets one tile of rows, so that x stays in the L2s (stream_once).
// ACT: the gated activation is compiled in: as a branch inside the one loop over the sums it made the epilogue of 256 x 256 tiles
// 13,000 instructions instead of 3,600, and the product 1 to 18 % slower (32 experts of 2,048 x 2,048 with 224 unequal rows 111 -> 91 us,
// 8 of 8,192 x 4,096 with 2,048 987 -> 940).
// 1,500 tokens with 6 of 48 experts (188 rows each), 2,048 x 4,096 with GELU and back, 32-bit results: 244 + 212 us -> 192 + 187 (x
// in pieces of 64 bytes, tiles of up to 256 rows and lookups between the stores before); 310 rows each 335 + 378 -> 280 + 296, 128
// rows 232 + 194 -> 169 + 166, 50 rows 182 + 158 -> 154 + 150, 750 rows 592 + 620 -> 560 + 584.  Gated, 8 experts of 4,096 x 4,096
// and back: 80 rows 158 + 84 -> 94 + 57, 2,048 rows 881 + 473 -> 862 + 463; 32 of 1,024 x 2,048 with 256 rows 79 + 52 -> 77 + 46.
// Tile order: the column tiles of a row tile follow each other, 32 in a row on one XCD.
#define GS_MAX_GROUPS 512
__device__ __forceinline__ float gelu_quick(float z) {
  // z erfc(-z / sqrt 2) / 2 with erfc(x) = t p(t) exp(-x^2), t = 1 / (1 + 0.4 x), p a polynomial fitted here to equal relative
  // errors for 0 <= x <= 7 (1.7e-7), for results that are rounded to bf16: the error function of the math library took a fifth
  // of a tile's time, with one wave a SIMD and nothing beside it.  Relative error over -9 .. 6, against 64 bits: at most 9e-6
  // (z (1 + erf) / 2, with its cancellation: 1e-3 at -4, all of the value from -6), and 5e-7 (2e-7) for |z| <= 1.
  const float x = fabsf(z) * 0.70710678118654752f, t = __builtin_amdgcn_rcpf(fmaf(0.4f, x, 1.f));
  float p = fmaf(0.0630790418f, t, -0.343721672f);
  p = fmaf(p, t, 0.58811212f), p = fmaf(p, t, -0.275384567f), p = fmaf(p, t, 0.349964476f);
  p = fmaf(p, t, 0.160084614f), p = fmaf(p, t, 0.232617782f), p = fmaf(p, t, 0.225248035f);
  const float q = 0.5f * p * t * __builtin_amdgcn_exp2f(-1.4426950408889634f * x * x);    // erfc(|z| / sqrt 2) / 2
  return z * (z < 0.f ? q : 1.f - q);
}

constexpr int NO_PAIR = -1;
template <int BM, int BN, bool F32, int ACT, bool ONCE>
__global__ void __launch_bounds__(256, 1) grouped_stream_kernel(GroupedArgs g, long a_bytes, long o_bytes) {
  constexpr int BK = 32, STAGES = stream_stages(BM, BN), PAIRS = stream_pairs(BM, BN), WAVES = 4;
  constexpr int XL = BM / 32, WL = BN / 64, PASSES = XL / 2 + WL;      // loads of a wave: of a pair of k-tiles of x, of a k-tile of W, a step
  constexpr int FM = BM / 32, FN = BN / 32;
  static_assert(FM == 4 || FM == 8, "row groups of a k-step");
  // A k-step of a wave goes row group by row group: 2 i + (its row of waves) is row group i's fragment of x, so that the waves share
  // what rows a tile has.  The first FMU groups always run, the others where the tile has rows for them, and in each the right
  // half of the columns where the tile has them; the loads lie in what always runs, since their number is what the waits count.
  constexpr int FMU = FM / 2, H = FN / 2, LOAD_EVERY = FMU * H / PASSES;
  constexpr unsigned FAR = 0x80000000u;            // beyond every view of x and W: read as zeros without traffic
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];      // x [PAIRS][BM][64], W [STAGES][BN][32]
  const int tid = threadIdx.x, lane = tid % SYN_WAVE, grid = (int)gridDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / SYN_WAVE);
  const int wr = wave / 2, wc = wave % 2;
  const int col_tiles = (g.N + BN - 1) / BN;
  // lane l of tiles_up_to[i]: the tiles of all segments up to 64 i + l (a prefix sum in every wave's registers, 64 segments at a time)
  constexpr int GROUP_PARTS = GS_MAX_GROUPS / SYN_WAVE;
  int tiles_up_to[GROUP_PARTS], all_rows = 0;
#pragma unroll
  for (int i = 0; i < GROUP_PARTS; ++i) {
    if (i * SYN_WAVE >= g.groups) {
      tiles_up_to[i] = all_rows;
      continue;
    }
    const int e = i * SYN_WAVE + lane;
    int n = e < g.groups ? (g.seg_start[e + 1] - g.seg_start[e] + BM - 1) / BM : 0;
#pragma unroll
    for (int off = 1; off < SYN_WAVE; off <<= 1) {
      const int o = __shfl_up(n, off, SYN_WAVE);
      if (lane >= off) n += o;
    }
    tiles_up_to[i] = all_rows + n;
    all_rows = __builtin_amdgcn_readlane(tiles_up_to[i], SYN_WAVE - 1);
  }
  // A last round that half of the workgroups could go round in is cut: each of its tiles becomes two of half the columns.
  const int all = all_rows * col_tiles;
  const int whole = all % grid * 2 <= grid ? all / grid * grid : all, tiles = 2 * all - whole;
  int at = ((int)blockIdx.x % 8) * (grid / 8) + (int)blockIdx.x / 8;
  if (at >= tiles) return;
  struct Tile {
    int e, row0, row_end, n0, columns, active;      // columns: BN or half of them; active: row groups that hold rows
  };
  auto tile_of = [&](int i) {
    const bool cut = i >= whole;
    const int half = cut ? (i - whole) % 2 : 0;
    if (cut) i = whole + (i - whole) / 2;
    const int rt = i / col_tiles;
    int lo = 0, first = 0;      // the segment and the tiles before it: those up to `lo` segments are no more than rt
#pragma unroll
    for (int p = 0; p < GROUP_PARTS; ++p) {
      const int n = p * SYN_WAVE < g.groups ? __builtin_popcountll(__ballot(tiles_up_to[p] <= rt)) : 0;
      if (n > 0) first = __builtin_amdgcn_readlane(tiles_up_to[p], n - 1);
      lo += n;
    }
    const int s0 = __builtin_amdgcn_readfirstlane(g.seg_start[lo]), s1 = __builtin_amdgcn_readfirstlane(g.seg_start[lo + 1]);
    // (the segment's tiles get the same number of rows, in steps of 32)
    const int n = (s1 - s0 + BM - 1) / BM, rows = ((s1 - s0 + n - 1) / n + 31) / 32 * 32;
    const int row0 = s0 + (rt - first) * rows, row_end = min(s1, row0 + rows), n0 = (i % col_tiles) * BN + half * (BN / 2);
    return Tile{lo, row0, row_end, n0, cut || g.N - n0 <= BN / 2 ? BN / 2 : BN, (row_end - row0 + 31) / 32};
  };
  const BufferView vx = buffer_view(g.a, (size_t)a_bytes);
  const size_t w_row = (size_t)g.K * sizeof(bf16);
  struct Rows {
    unsigned at[XL];      // offsets of the lane's pieces of rows: load p of x takes 128 bytes of tile rows (p * WAVES + wave) * 8 .. + 8
  };
  auto rows_of = [&](const Tile& t) {
    Rows x;
    const int r0 = t.row0 + wave * 8 + lane / 8;
    int row[XL];
#pragma unroll
    for (int p = 0; p < XL; ++p) row[p] = min(r0 + p * WAVES * 8, t.row_end - 1);
    if (g.a_rows) {      // (asked for together)
#pragma unroll
      for (int p = 0; p < XL; ++p) row[p] = g.a_rows[row[p]];
    }
#pragma unroll
    for (int p = 0; p < XL; ++p)
      x.at[p] = r0 + p * WAVES * 8 < t.row_end ? (unsigned)((size_t)row[p] * g.lda * sizeof(bf16)) + ((lane % 8) ^ (wave % 2 * 4 + lane / 16)) * 16 : FAR;
    return x;
  };
  auto weights_of = [&](const Tile& t) {
    return buffer_view((const bf16*)g.w + (size_t)t.e * g.w_group + (size_t)t.n0 * g.K, (size_t)max(0, min(t.columns, g.N - t.n0)) * w_row);
  };
  unsigned src_w[WL];
#pragma unroll
  for (int p = 0; p < WL; ++p) src_w[p] = (unsigned)((size_t)(p * WAVES + wave) * 16 * w_row + lane * 16);
  // where the loads have got to, as in gemm_stream_kernel
  constexpr int W_TILE = BK * (int)sizeof(bf16) * 16, X_PAIR = 2 * BK * (int)sizeof(bf16);
  constexpr int W_BUF = BN * BK * (int)sizeof(bf16), X_BUF = BM * X_PAIR;
  const int steps = g.K / BK, w_end = steps * W_TILE, x_end = steps * (X_PAIR / 2);
  const int x_to = wave * 8 * X_PAIR, w_to = PAIRS * X_BUF + wave * 16 * BK * (int)sizeof(bf16);
  int x_way = 0, w_way = 0;
  Rows x_rows, x_rows_then;
  BufferView w_view, w_then;
  auto onward_w = [&] {
    w_way += W_TILE;
    if (__builtin_expect(w_way == w_end, 0)) w_way = 0, w_view = w_then;
  };
  auto onward_x = [&] {
    x_way += X_PAIR;
    if (__builtin_expect(x_way == x_end, 0)) x_way = 0, x_rows = x_rows_then;
  };
  auto fetch_x = [&](int xbuf, int p) {
    buffer_to_lds16(vx, (char*)smem + xbuf + x_to + p % XL * (WAVES * 8 * X_PAIR), x_rows.at[p % XL], x_way);
  };
  auto fetch_w = [&](int buf, int p) {
    buffer_to_lds16<ONCE>(w_view, (char*)smem + buf + w_to + p * (WAVES * 16 * BK * (int)sizeof(bf16)), src_w[p], w_way);
  };
  f32x4 acc[FM][FN];
  const int r16 = lane % 16, q4 = lane / 16;
  // in bytes; the second k-tile of a pair: chunks 4 to 7, bit 2 of the slot
  const int x_at = ((16 * wr + r16) * 2 * BK + (q4 ^ (r16 / 2)) * 8) * 2, x_at2 = x_at ^ 64;
  bf16x8 a[2][FM], b[2][FN];
  auto read_x = [&](int xbuf, int half, int set, int i) { a[set][i] = *(const bf16x8*)((const char*)smem + xbuf + (half ? x_at2 : x_at) + i * 32 * X_PAIR); };
  auto read_w = [&](int buf, int set, int j, int w_at) { b[set][j] = *(const bf16x8*)((const char*)smem + buf + w_at + j * 16 * BK * 2); };
  int buf = 0, xbuf = 0, xbuf_before = STAGES / 2 * X_BUF;
  auto step = [&](int parts, int w_at, auto set, auto fresh) {
    constexpr int SET = decltype(set)::value;
    const int next = buf + W_BUF == STAGES * W_BUF ? 0 : buf + W_BUF;
    const int xnext = SET ? (xbuf + X_BUF == PAIRS * X_BUF ? 0 : xbuf + X_BUF) : xbuf;
    // four matrix instructions of row group I from column J on, passed over as a whole where bit 2 I + J / H of `parts` is clear: the
    // branch stands inside the statement, so that the sums stay where they are (around statements the compiler moved them)
    auto four = [&](auto group, auto column) {
      constexpr int I = decltype(group)::value, J = decltype(column)::value, BIT = 2 * I + J / H;
      if constexpr (decltype(fresh)::value)
        asm volatile("s_bitcmp1_b32 %9, %10\n\ts_cbranch_scc0 .Lpast%=\n\t"
                     "v_mfma_f32_16x16x32_bf16 %0, %4, %8, 0\n\tv_mfma_f32_16x16x32_bf16 %1, %5, %8, 0\n\t"
                     "v_mfma_f32_16x16x32_bf16 %2, %6, %8, 0\n\tv_mfma_f32_16x16x32_bf16 %3, %7, %8, 0\n.Lpast%=:"
                     : "=a"(acc[I][J]), "=a"(acc[I][J + 1]), "=a"(acc[I][J + 2]), "=a"(acc[I][J + 3])
                     : "v"(b[SET][J]), "v"(b[SET][J + 1]), "v"(b[SET][J + 2]), "v"(b[SET][J + 3]), "v"(a[SET][I]), "s"(parts), "n"(BIT) : "scc");
      else
        asm volatile("s_bitcmp1_b32 %9, %10\n\ts_cbranch_scc0 .Lpast%=\n\t"
                     "v_mfma_f32_16x16x32_bf16 %0, %4, %8, %0\n\tv_mfma_f32_16x16x32_bf16 %1, %5, %8, %1\n\t"
                     "v_mfma_f32_16x16x32_bf16 %2, %6, %8, %2\n\tv_mfma_f32_16x16x32_bf16 %3, %7, %8, %3\n.Lpast%=:"
                     : "+a"(acc[I][J]), "+a"(acc[I][J + 1]), "+a"(acc[I][J + 2]), "+a"(acc[I][J + 3])
                     : "v"(b[SET][J]), "v"(b[SET][J + 1]), "v"(b[SET][J + 2]), "v"(b[SET][J + 3]), "v"(a[SET][I]), "s"(parts), "n"(BIT) : "scc");
      __builtin_amdgcn_sched_barrier(0);
    };
    auto row_group = [&](auto group) {
      constexpr int I = decltype(group)::value;
      if constexpr (I < FMU) {
#pragma unroll
        for (int j = 0; j < H; ++j) {
          if constexpr (decltype(fresh)::value)
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[I][j]) : "v"(b[SET][j]), "v"(a[SET][I]));
          else
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[I][j]) : "v"(b[SET][j]), "v"(a[SET][I]));
          const int q = I * H + j;
          if (q % LOAD_EVERY == 0 && q / LOAD_EVERY < PASSES) {
            const int p = q / LOAD_EVERY;
            if (p < XL / 2) fetch_x(SET ? xbuf : xbuf_before, SET ? p : p + XL / 2);
            else fetch_w(buf, p - XL / 2);
          }
          if (q % FMU == FMU - 1) read_w(next, SET ^ 1, q / FMU, w_at);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        four(group, std::integral_constant<int, 0>{});
      }
      read_x(xnext, SET ^ 1, SET ^ 1, I);
      __builtin_amdgcn_sched_barrier(0);
      four(group, std::integral_constant<int, H>{});
      if constexpr (I < FMU) {
#pragma unroll
        for (int j = H + I * H / FMU; j < H + (I + 1) * H / FMU; ++j) read_w(next, SET ^ 1, j, w_at);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    row_group(std::integral_constant<int, 0>{}), row_group(std::integral_constant<int, 1>{});
    row_group(std::integral_constant<int, 2>{}), row_group(std::integral_constant<int, 3>{});
    if constexpr (FM > 4) {
      row_group(std::integral_constant<int, 4>{}), row_group(std::integral_constant<int, 5>{});
      row_group(std::integral_constant<int, 6>{}), row_group(std::integral_constant<int, 7>{});
    }
    onward_w();
    if constexpr (SET == 0) onward_x();
    else xbuf_before = xbuf, xbuf = xnext;
    buf = next;
  };
  constexpr int YOUNGER = (STAGES - 2) * PASSES;
  auto landed = [&] {
    __builtin_amdgcn_s_waitcnt(0x0070 | (YOUNGER & 15) | ((YOUNGER >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  Tile t = tile_of(at);
  bool more = at + grid < tiles;
  Tile t_next = more ? tile_of(at + grid) : t;       // (behind the last tile: loads that nobody reads)
  x_rows = rows_of(t), w_view = weights_of(t);
  x_rows_then = rows_of(t_next), w_then = weights_of(t_next);
  __builtin_amdgcn_s_waitcnt(0x0070);        // (the row lists' own loads: the counts below are those of the rings alone)
  __builtin_amdgcn_sched_barrier(0);
  // what the steps before the first would have asked for
#pragma unroll
  for (int p = 0; p < XL / 2; ++p) fetch_x(0, p);
#pragma unroll
  for (int s = 0; s < STAGES; ++s) {
#pragma unroll
    for (int p = 0; p < XL / 2; ++p) fetch_x((s + 1) / 2 * X_BUF, s % 2 ? p : p + XL / 2);
#pragma unroll
    for (int p = 0; p < WL; ++p) fetch_w(s * W_BUF, p);
    onward_w();
    if (s % 2 == 0) onward_x();
  }
  landed();
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  const BufferView vo = buffer_view(g.out, (size_t)o_bytes);
  for (;;) {
    const int active = t.active, wn = wc * (t.columns / 2), w_at = PAIRS * X_BUF + (wn * BK + lane * 8) * 2;
    const bool wide = t.columns == BN;
    // bit 2 i: row group i holds rows, bit 2 i + 1: and the tile its right half of columns
    const int parts = ((1 << 2 * active) - 1) & (wide ? 0xffff : 0x5555);
    // the first fragments: all of them, the tile before may have had fewer rows or columns
#pragma unroll
    for (int i = 0; i < FM; ++i) read_x(xbuf, 0, 0, i);
#pragma unroll
    for (int j = 0; j < FN; ++j) read_w(buf, 0, j, w_at);
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): they are in registers,
    __builtin_amdgcn_s_barrier();         // everywhere
    __builtin_amdgcn_sched_barrier(0);
    step(parts, w_at, Even{}, std::true_type{}), landed();
    step(parts, w_at, Odd{}, std::false_type{}), landed();
    // (entered always, K >= 256: with a way round the loop the compiler carried some sums of the 256-row tile through vector
    // registers there, read right behind matrix instructions that it does not know for such)
    int kt = 2;
    do {
      step(parts, w_at, Even{}, std::false_type{}), landed();
      step(parts, w_at, Odd{}, std::false_type{}), landed();
      kt += 2;
    } while (kt < steps);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");     // (see gemm_stream_kernel)
    __builtin_amdgcn_sched_barrier(0);
    // What the stores look up, and the rows of the tile after the next: all of it before the first store, since whatever is loaded
    // behind stores is waited for behind them too.
    const int r0 = t.row0 + 16 * wr + r16;
    int o_row[FM];
    float weight_of[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) o_row[i] = min(r0 + 32 * i, t.row_end - 1), weight_of[i] = 1.f;
    if (g.row_weight) {
#pragma unroll
      for (int i = 0; i < FM; ++i) weight_of[i] = g.row_weight[o_row[i]];
    }
    if (g.o_rows) {
#pragma unroll
      for (int i = 0; i < FM; ++i) o_row[i] = g.o_rows[o_row[i]];
    }
    const bool more_then = more && at + 2 * grid < tiles;
    const Tile t_then = more_then ? tile_of(at + 2 * grid) : t_next;
    const Rows rows_then = rows_of(t_then);
    __builtin_amdgcn_sched_barrier(0);
    // lane: row t.row0 + 32 i + 16 wr + r16, columns t.n0 + wn + 16 j + 4 q4 .. + 4
    auto store_all = [&](auto of) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if (i >= FMU && i >= active) break;
        const unsigned row = (unsigned)((size_t)o_row[i] * g.ldo * (F32 ? 4 : 2));
        const bool in = r0 + 32 * i < t.row_end;
        const float weight = weight_of[i];
#pragma unroll
        for (int j = 0; j < FN; ++j) asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int n = t.n0 + wn + 16 * j + 4 * q4;
          const bool ok = in && n < g.N && (j < H || wide);
          if constexpr (ACT != NO_PAIR) {
            const float v0 = of(acc[i][j][0], acc[i][j][1]) * weight, v1 = of(acc[i][j][2], acc[i][j][3]) * weight;
            if constexpr (F32) {
              buffer_store4(vo, v0, ok ? row + (n / 2) * 4 : SYN_NOWHERE);
              buffer_store4(vo, v1, ok ? row + (n / 2) * 4 + 4 : SYN_NOWHERE);
            } else {
              typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
              buffer_store4(vo, __builtin_bit_cast(float, bf16x2{(bf16)v0, (bf16)v1}), ok ? row + (n / 2) * 2 : SYN_NOWHERE);
            }
          } else {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = of(acc[i][j][e], 0.f) * weight;
            if constexpr (F32) {
              buffer_store16(vo, __builtin_bit_cast(u32x4, v), ok ? row + n * 4 : SYN_NOWHERE, 0);
            } else {
              bf16x4 h;
#pragma unroll
              for (int e = 0; e < 4; ++e) h[e] = (bf16)v[e];
              buffer_store8(vo, __builtin_bit_cast(u32x2, h), ok ? row + n * 2 : SYN_NOWHERE);
            }
          }
        }
      }
    };
    if constexpr (ACT != NO_PAIR) {
      store_all([&](float gt, float up) { return gated_quick<ACT, F32>(gt, up, g.limit); });
    } else {
      if (g.act == 0) store_all([&](float v, float) { return v; });
      else if (g.act == 2) store_all([&](float v, float) { return point_activation(SYN_POINT_RELU_SQUARED, v); });
      else store_all([&](float v, float) { return gelu_quick(v); });
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!more) break;
    at += grid, t = t_next, t_next = t_then, more = more_then;
    x_rows_then = rows_then, w_then = weights_of(t_next);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
}

template <int BM, bool F32, int ACT, bool ONCE>
static int launch_grouped_stream(const GroupedArgs& g, long a_bytes, long o_bytes, hipStream_t stream) {
  constexpr int BN = 256;
  const size_t lds = stream_lds(BM, BN);
  static OncePerDevice raised;
  const hipError_t e = once_per_device(raised, [&] {
    return hipFuncSetAttribute((const void*)grouped_stream_kernel<BM, BN, F32, ACT, ONCE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  });
  SYN_CHECK(e == hipSuccess, "grouped_product: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
  grouped_stream_kernel<BM, BN, F32, ACT, ONCE><<<syn_compute_units() / 8 * 8, 256, lds, stream>>>(g, a_bytes, o_bytes);
  return 0;
}
template <bool F32, int ACT>
static int launch_grouped_stream_as(int rows, bool once, const GroupedArgs& g, long a_bytes, long o_bytes, hipStream_t stream) {
  if (rows == 128) return launch_grouped_stream<128, F32, ACT, true>(g, a_bytes, o_bytes, stream);
  if (once) return launch_grouped_stream<256, F32, ACT, true>(g, a_bytes, o_bytes, stream);
  return launch_grouped_stream<256, F32, ACT, false>(g, a_bytes, o_bytes, stream);
}
template <int ACT>
static int launch_grouped_stream_for(int rows, bool once, const GroupedArgs& g, long a_bytes, long o_bytes, hipStream_t stream) {
  return g.out_is_f32 ? launch_grouped_stream_as<true, ACT>(rows, once, g, a_bytes, o_bytes, stream)
                      : launch_grouped_stream_as<false, ACT>(rows, once, g, a_bytes, o_bytes, stream);
}

// Rows of a streamed tile, and whether W's loads are marked non-temporal, from what the host knows: the rows a segment has on average.
// A tile leaves out the rows that its segment does not have, so the higher one costs little where there are few, while a segment of two
// tiles brings in W twice: against the best of 64, 128 and 256 with equal and unequal segments, 50 rows on average 1.01, 1.02 and 1.06
// and 1.10, 1.02 and 1.07 times as long, 80 rows 1.52, 1.01, 1.04 and 1.44, 1.01, 1.04, 100 rows 1.42, 1.01, 1.04 and 1.63, 1.19, 1.01, 128 rows 1.37,
// 1.01, 1.04 and 1.80, 1.31, 1.00.  Tiles of 64 rows won 6 % at most (8 experts with 50 rows each).
// Non-temporal loads against plain ones, gated products and the others: equal segments of 50 to 188 rows -7 and -6 %, 224 rows -5 and -7,
// 310 and more +2 to 5 and +1 to 3; unequal ones (0.4 to 1.6 times the average) -4 to 7 and -3 to 5 %, with 224 rows +2 and 0, 256 +4 and 0, more
// +4 and +5.
// All of it over 184 products of 8 to 128 experts, 768 to 28,672 wide, with 50 to 2,048 rows a segment: what this picks takes 1.6 % longer than
// the best of the six on average, 4 % of them lose more than 10, 1.32 times as long at the worst (8 experts with 400 unequal rows, whose
// tiles just exceed a round).
static int stream_rows(long rows_a_group) { return rows_a_group <= 80 ? 128 : 256; }
static bool stream_once(long rows_a_group) { return rows_a_group <= 224; }
// (for tests of the rules)
SYN_EXPORT int syn_grouped_stream_rows(int rows_a_group) { return stream_rows(rows_a_group); }
SYN_EXPORT int syn_grouped_stream_once(int rows_a_group) { return stream_once(rows_a_group); }

// rows_bound: with segments, the number of rows in all segments together (what the index lists hold)
// a_total, o_total: rows that a and out hold
SYN_EXPORT int syn_grouped_product(const void* a, long lda, long a_group, const void* w, long w_group, long ldw, void* out,
                                   long ldo, long o_group, int in_is_f32, int out_is_f32, const int* seg_start,
                                   const int* a_rows, const int* o_rows, const float* row_weight, const float* gate,
                                   long gate_ld, long gate_group, int gate_col, int act, int M, int N, int K, int groups,
                                   int rows_bound, int force_simt, int w_packed, int pair, float limit, long a_total,
                                   long o_total, hipStream_t stream) {
  SYN_CHECK(M > 0 && N > 0 && K > 0 && groups > 0, "grouped_product: empty input (%d rows, %d x %d, %d groups)", M, N, K, groups);
  SYN_CHECK(act >= 0 && act <= 2, "grouped_product: unknown activation code %d", act);
  SYN_CHECK(pair >= 0 && pair <= SYN_ACT_COUNT && (pair == 0 || (N % 2 == 0 && act == 0 && gate == nullptr)),
            "grouped_product: a gated activation (code %d) over %d rows of W in pairs, with no other activation", pair - 1, N);
  SYN_CHECK(seg_start != nullptr || (a_rows == nullptr && o_rows == nullptr && row_weight == nullptr),
            "grouped_product: index lists and row weights come with segments");
  SYN_CHECK(seg_start == nullptr || rows_bound > 0, "grouped_product: segments over %d rows", rows_bound);
  SYN_CHECK(seg_start == nullptr || gate == nullptr, "grouped_product: a gate is read by row and group, not through segments");
  SYN_CHECK(!w_packed || (!in_is_f32 && N % 16 == 0 && K % 32 == 0),
            "grouped_product: matrices in fragment order are bf16 of %d x %d (multiples of 16 and 32)?", N, K);
  const GroupedArgs g = {a, lda, a_group, w, w_group, ldw, out, ldo, o_group, out_is_f32, seg_start, a_rows, o_rows,
                         row_weight, gate, gate_ld, gate_group, gate_col, act, pair, limit, M, N, K, groups, w_packed};
  const bool aligned = K % 32 == 0 && lda % 8 == 0 && a_group % 8 == 0 && ldw % 8 == 0 && w_group % 8 == 0 &&
                       (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0;
  // many rows a group (on average, where the host does not know the segments): the tiles through LDS
  const long rows_a_group = seg_start ? rows_bound / groups : M;
  const bool chunks = K % 8 == 0 && lda % 8 == 0 && a_group % 8 == 0 && ldw % 8 == 0 && w_group % 8 == 0 &&
                      (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0;
  // the streamed tiles: W in fragment order, K in pairs of k-steps and a ring of them (eight) at least, 16-byte stores, and
  // offsets of x and out that fit 31 and 32 bits (a GELU is stored as bf16 there: gelu_quick)
  const long a_bytes = a_total * lda * 2, o_bytes = o_total * ldo * (out_is_f32 ? 4 : 2);
  const bool streamed = seg_start && w_packed && chunks && force_simt == 0 && rows_a_group >= 48 && K % 64 == 0 && K >= 256 &&
                        groups <= GS_MAX_GROUPS && N % 32 == 0 && ldo % 8 == 0 && (uintptr_t)out % 16 == 0 && ldw == K &&
                        a_total > 0 && o_total > 0 && a_bytes < (1L << 31) && o_bytes < (1L << 32) - 16 &&
                        (long)N * K * 2 < (1L << 31) && !(act == 1 && out_is_f32);
  if (streamed) {
    const int rows = stream_rows(rows_a_group);
    const bool once = stream_once(rows_a_group);
    int rc;
    if (!pair) rc = launch_grouped_stream_for<NO_PAIR>(rows, once, g, a_bytes, o_bytes, stream);
    else if (pair - 1 == SYN_ACT_SILU) rc = launch_grouped_stream_for<SYN_ACT_SILU>(rows, once, g, a_bytes, o_bytes, stream);
    else if (pair - 1 == SYN_ACT_SWIGLU_LIMIT) rc = launch_grouped_stream_for<SYN_ACT_SWIGLU_LIMIT>(rows, once, g, a_bytes, o_bytes, stream);
    else rc = launch_grouped_stream_for<SYN_ACT_GELU_TANH>(rows, once, g, a_bytes, o_bytes, stream);
    if (rc) return rc;
  } else if (!in_is_f32 && chunks && force_simt == 0 && rows_a_group >= 48) {
    const int row_tiles = seg_start ? (rows_bound + GT_BM - 1) / GT_BM + groups : (M + GT_BM - 1) / GT_BM;
    const int places = (row_tiles * ((N + GT_BN - 1) / GT_BN) + 7) / 8 * 8;
    const dim3 grid(places, 1, seg_start ? 1 : groups);
    const size_t lds = (size_t)2 * (GT_BM + GT_BN) * GT_LD * sizeof(bf16);
    static OncePerDevice raised;
    const hipError_t e = once_per_device(raised, [&] {
      const hipError_t r = hipFuncSetAttribute((const void*)grouped_product_tiled_kernel<false>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      return r != hipSuccess ? r : hipFuncSetAttribute((const void*)grouped_product_tiled_kernel<true>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    SYN_CHECK(e == hipSuccess, "grouped_product: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
    if (pair) grouped_product_tiled_kernel<true><<<grid, 256, lds, stream>>>(g);
    else grouped_product_tiled_kernel<false><<<grid, 256, lds, stream>>>(g);
  } else if (!in_is_f32 && aligned && force_simt != 1) {
    const int row_tiles = seg_start ? (rows_bound + GP_TM - 1) / GP_TM + groups : (M + GP_TM - 1) / GP_TM;
    const long wide = (long)row_tiles * ((N + 255) / 256) * (seg_start ? 1 : groups);
    // (force_simt 3: the wide waves whatever the sizes, for tests)
    if (wide >= 8L * syn_compute_units() || force_simt == 3) {
      const dim3 grid(row_tiles, (N + 255) / 256, seg_start ? 1 : groups);
      grouped_product_mfma_kernel<4><<<grid, 256, 0, stream>>>(g);
    } else {
      const dim3 grid(row_tiles, (N + 63) / 64, seg_start ? 1 : groups);
      grouped_product_mfma_kernel<1><<<grid, 256, 0, stream>>>(g);
    }
  } else {
    const dim3 grid(seg_start ? rows_bound : M, (N + 31) / 32, seg_start ? 1 : groups);
    if (in_is_f32) grouped_product_simt_kernel<float><<<grid, 256, 0, stream>>>(g);
    else grouped_product_simt_kernel<bf16><<<grid, 256, 0, stream>>>(g);
  }
  SYN_LAUNCH_CHECK("grouped_product");
  return 0;
}

// ---------------------------------------------------------------- router: the largest `top` logits, their softmax
// One wave a token over its row of logits z [E] (32-bit sums of a product that ran before, or `parts` partial sums of them, added
// here) + bias; of equal logits the lower index comes first.
#define ROUTE_MAX_EXPERTS 1024
#define ROUTE_MAX_TOP 64
__global__ void __launch_bounds__(256) route_topk_kernel(const float* __restrict__ logits, const float* __restrict__ bias,
                                                         int* __restrict__ ids, float* __restrict__ weights,
                                                         int n_tokens, int E, int top, int parts) {
  __shared__ float zs[4][ROUTE_MAX_EXPERTS];
  __shared__ float chosen_s[4][ROUTE_MAX_TOP];
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE, tok = blockIdx.x * 4 + wave;
  if (tok >= n_tokens) return;             // (waves work alone: no barrier of the workgroup below)
  float* z = zs[wave];
  float* chosen = chosen_s[wave];
  for (int e = lane; e < E; e += SYN_WAVE) {
    const float* at = logits + (size_t)tok * E + e;
    const size_t step = (size_t)n_tokens * E;
    float sum = at[0];
#pragma unroll 8
    for (int p = 1; p < parts; ++p) sum += at[p * step];
    z[e] = sum + (bias ? bias[e] : 0.f);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int t = 0; t < top; ++t) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < E; e += SYN_WAVE) {
      const float v = z[e];
      if (v > best) best = v, at = e;      // (a lane meets its experts in rising order)
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, SYN_WAVE);
      const int oa = __shfl_xor(at, off, SYN_WAVE);
      if (ob > best || (ob == best && oa < at)) best = ob, at = oa;
    }
    if (lane == 0) {
      if (at >= E) at = t;          // every logit left is NaN or -inf: any expert, and no access beyond the table
      ids[(size_t)tok * top + t] = at;
      chosen[t] = best;
      z[at] = -INFINITY;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  if (lane == 0) {
    const float m = chosen[0];      // the first chosen is the largest
    float sum = 0.f;
    for (int t = 0; t < top; ++t) sum += expf(chosen[t] - m);
    for (int t = 0; t < top; ++t) weights[(size_t)tok * top + t] = expf(chosen[t] - m) / sum;
  }
}

SYN_EXPORT int syn_route_topk(const float* logits, const float* bias, int* ids, float* weights, int n_tokens, int E,
                              int top, int parts, hipStream_t stream) {
  SYN_CHECK(n_tokens > 0 && parts > 0, "route_topk: empty input");
  SYN_CHECK(E > 0 && E <= ROUTE_MAX_EXPERTS, "route_topk: %d experts (at most %d)", E, ROUTE_MAX_EXPERTS);
  SYN_CHECK(top > 0 && top <= E && top <= ROUTE_MAX_TOP, "route_topk: the %d largest of %d (at most %d)", top, E, ROUTE_MAX_TOP);
  route_topk_kernel<<<(n_tokens + 3) / 4, 256, 0, stream>>>(logits, bias, ids, weights, n_tokens, E, top, parts);
  SYN_LAUNCH_CHECK("route_topk");
  return 0;
}

// ---------------------------------------------------------------- a router that scores all experts
// s = softmax(logits) over all E outputs, or, with `sigmoid`, the sigmoid of each (32-bit).  The choice is made on
// s + correction: the E outputs form n_groups equal groups of neighbours, a group's score is its largest choice score, or,
// with group_two, the sum of its two largest; only members of the keep_groups best groups
// can be chosen (the others count as minus infinity), and of those the `top` largest are taken (the lower index of
// equal ones, for groups and for experts).  weights: the chosen experts' s itself, without the correction; renorm:
// divided by their sum (+ renorm_eps).  One wave a token.
__global__ void __launch_bounds__(256) route_scores_kernel(const float* __restrict__ logits, const float* __restrict__ correction,
                                                           int* __restrict__ ids, float* __restrict__ weights, int n_tokens,
                                                           int E, int ld, int top, int n_groups, int keep_groups, int renorm,
                                                           float scale, int sigmoid, int group_two, float renorm_eps) {
  __shared__ float ss[4][ROUTE_MAX_EXPERTS];       // the scores
  __shared__ float cs[4][ROUTE_MAX_EXPERTS];       // the choice scores
  __shared__ float gs[4][ROUTE_MAX_EXPERTS];       // the groups' scores
  __shared__ float chosen_s[4][ROUTE_MAX_TOP];
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE, tok = blockIdx.x * 4 + wave;
  if (tok >= n_tokens) return;             // (waves work alone: no barrier of the workgroup below)
  float* sc = ss[wave];
  float* c = cs[wave];
  float* grp = gs[wave];
  float* chosen = chosen_s[wave];
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  float sum = 1.f;
  if (sigmoid) {
    for (int e = lane; e < E; e += SYN_WAVE) sc[e] = 1.f / (1.f + expf(-logits[(size_t)tok * ld + e]));
  } else {
    float mx = -INFINITY;
    for (int e = lane; e < E; e += SYN_WAVE) mx = fmaxf(mx, logits[(size_t)tok * ld + e]);
    mx = wave_max(mx);
    sum = 0.f;
    for (int e = lane; e < E; e += SYN_WAVE) {
      const float p = expf(logits[(size_t)tok * ld + e] - mx);
      sc[e] = p;
      sum += p;
    }
    sum = wave_sum(sum);
  }
  const int per = E / n_groups;
  for (int e = lane; e < E; e += SYN_WAVE) {
    sc[e] = sc[e] / sum;
    c[e] = sc[e] + (correction ? correction[e] : 0.f);
  }
  wave_sync();
  if (keep_groups < n_groups) {
    for (int g = lane; g < n_groups; g += SYN_WAVE) {
      float best = -INFINITY, second = -INFINITY;
      for (int j = 0; j < per; ++j) {
        const float v = c[g * per + j];
        second = fmaxf(second, fminf(best, v));
        best = fmaxf(best, v);
      }
      grp[g] = group_two && per > 1 ? best + second : best;
    }
    wave_sync();
    // a group stays if fewer than keep_groups others come before it (a larger score, or an equal one at a lower index)
    for (int g = lane; g < n_groups; g += SYN_WAVE) {
      int before = 0;
      for (int o = 0; o < n_groups; ++o) before += (grp[o] > grp[g] || (grp[o] == grp[g] && o < g)) ? 1 : 0;
      if (before >= keep_groups)
        for (int j = 0; j < per; ++j) c[g * per + j] = -INFINITY;
    }
    wave_sync();
  }
  for (int t = 0; t < top; ++t) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < E; e += SYN_WAVE) {
      const float v = c[e];
      if (v > best) best = v, at = e;      // (a lane meets its experts in rising order)
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, SYN_WAVE);
      const int oa = __shfl_xor(at, off, SYN_WAVE);
      if (ob > best || (ob == best && oa < at)) best = ob, at = oa;
    }
    if (lane == 0) {
      if (at >= E) at = t;          // nothing left to choose from: any expert, and no access beyond the table
      ids[(size_t)tok * top + t] = at;
      chosen[t] = sc[at];
      c[at] = -INFINITY;
    }
    wave_sync();
  }
  if (lane == 0) {
    float total = 1.f;
    if (renorm) {
      total = 0.f;
      for (int t = 0; t < top; ++t) total += chosen[t];
      total += renorm_eps;
    }
    for (int t = 0; t < top; ++t) weights[(size_t)tok * top + t] = chosen[t] / total * scale;
  }
}

// logits: rows of `ld` values whose first E are the router's outputs; weights: the chosen scores (over their sum with
// renorm) times `scale`
SYN_EXPORT int syn_route_scores(const float* logits, const float* correction, int* ids, float* weights, int n_tokens, int E,
                                int ld, int top, int n_groups, int keep_groups, int renorm, float scale, int sigmoid, int group_two,
                                float renorm_eps, hipStream_t stream) {
  SYN_CHECK(ld >= E, "route_scores: rows of %d values for %d experts", ld, E);
  SYN_CHECK(n_tokens > 0, "route_scores: empty input");
  SYN_CHECK(E > 0 && E <= ROUTE_MAX_EXPERTS, "route_scores: %d experts (at most %d)", E, ROUTE_MAX_EXPERTS);
  SYN_CHECK(n_groups > 0 && E % n_groups == 0 && keep_groups > 0 && keep_groups <= n_groups,
            "route_scores: %d experts in %d groups of which %d stay", E, n_groups, keep_groups);
  SYN_CHECK(top > 0 && top <= ROUTE_MAX_TOP && top <= keep_groups * (E / n_groups),
            "route_scores: the %d largest of %d groups of %d (at most %d)", top, keep_groups, E / n_groups, ROUTE_MAX_TOP);
  route_scores_kernel<<<(n_tokens + 3) / 4, 256, 0, stream>>>(logits, correction, ids, weights, n_tokens, E, ld, top, n_groups,
                                                             keep_groups, renorm, scale, sigmoid, group_two, renorm_eps);
  SYN_LAUNCH_CHECK("route_scores");
  return 0;
}

// Experts that are the identity: for the places r of seg_start[first] .. seg_start[last] (the segments of the experts
// first .. last - 1 after the sort), out[o_rows[r]] = weight_of[r] * x[a_rows[r]].  x [*, H] in the engine's type, out
// [*, H] float.  One workgroup a place of the list; those outside the range leave at once.
template <typename T>
__global__ void __launch_bounds__(256) route_identity_kernel(const T* __restrict__ x, float* __restrict__ out,
                                                             const int* __restrict__ seg_start, int first, int last,
                                                             const int* __restrict__ a_rows, const int* __restrict__ o_rows,
                                                             const float* __restrict__ weight_of, int H) {
  const int r = blockIdx.x;
  if (r < seg_start[first] || r >= seg_start[last]) return;
  const T* src = x + (size_t)a_rows[r] * H;
  float* dst = out + (size_t)o_rows[r] * H;
  const float w = weight_of[r];
  for (int i = threadIdx.x; i < H; i += blockDim.x) dst[i] = w * to_f32<T>(src[i]);
}

SYN_EXPORT int syn_route_identity(const void* x, int is_f32, float* out, const int* seg_start, int first, int last,
                                  const int* a_rows, const int* o_rows, const float* weight_of, int places, int H,
                                  hipStream_t stream) {
  SYN_CHECK(places > 0 && H > 0 && first >= 0 && last >= first, "route_identity: empty input");
  if (last == first) return 0;
  if (is_f32)
    route_identity_kernel<float><<<places, 256, 0, stream>>>((const float*)x, out, seg_start, first, last, a_rows, o_rows,
                                                             weight_of, H);
  else
    route_identity_kernel<bf16><<<places, 256, 0, stream>>>((const bf16*)x, out, seg_start, first, last, a_rows, o_rows,
                                                            weight_of, H);
  SYN_LAUNCH_CHECK("route_identity");
  return 0;
}

// ---------------------------------------------------------------- the router's choices as segments
// P = n_tokens * top pairs (token n, its t-th expert), pair p = n * top + t.  Sorted by expert:
//   seg_start[e] .. seg_start[e + 1]: the places of expert e;  for a place r:
//   tok_of[r] = n, pair_of[r] = p, part_of[r] = t * n_tokens + n (the pair's row in partial sums [top, n_tokens]),
//   weight_of[r] = weights[p].
// The order inside a segment is the order of arrival; no result depends on it (a row's sums do not depend on its place in a tile).
// What bounds it: the lists are written 4 bytes at a time all over, 64 lines a store of a wave, so the pairs are spread over workgroups;
// each counts all pairs and those in front of its own, which gives it its places without a word to the others.  9,000 pairs, 48
// experts: 23 -> 8.7 us.
#define SORT_PAIRS 1024      // of a workgroup, at least
#define SORT_GROUPS 64
__global__ void __launch_bounds__(1024) route_sort_kernel(const int* __restrict__ ids, const float* __restrict__ weights,
                                                          int* __restrict__ seg_start, int* __restrict__ tok_of,
                                                          int* __restrict__ pair_of, int* __restrict__ part_of,
                                                          float* __restrict__ weight_of, int n_tokens, int top, int E, int share) {
  __shared__ int count[ROUTE_MAX_EXPERTS], earlier[ROUTE_MAX_EXPERTS], wave_n[16];
  const int P = n_tokens * top, tid = threadIdx.x, lane = tid % SYN_WAVE, wave = tid / SYN_WAVE;
  const int lo = blockIdx.x * share, hi = min(P, lo + share);
  static_assert(ROUTE_MAX_EXPERTS <= 1024, "a thread an expert");
  count[tid] = 0, earlier[tid] = 0;
  __syncthreads();
  for (int p = tid; p < P; p += blockDim.x) {
    const int e = min(max(ids[p], 0), E - 1);
    atomicAdd(&count[e], 1);
    if (p < lo) atomicAdd(&earlier[e], 1);
  }
  __syncthreads();
  // the places before each expert's: a prefix sum over the threads
  const int own = count[tid];
  int upto = own;
#pragma unroll
  for (int off = 1; off < SYN_WAVE; off <<= 1) {
    const int o = __shfl_up(upto, off, SYN_WAVE);
    if (lane >= off) upto += o;
  }
  if (lane == SYN_WAVE - 1) wave_n[wave] = upto;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; ++w) upto += w < wave ? wave_n[w] : 0;
  earlier[tid] += upto - own;      // the expert's next place for this workgroup
  if (blockIdx.x == 0) {
    if (tid < E) seg_start[tid] = upto - own;
    if (tid == E - 1) seg_start[E] = upto;
  }
  __syncthreads();
  for (int p = lo + tid; p < hi; p += blockDim.x) {
    const int r = atomicAdd(&earlier[min(max(ids[p], 0), E - 1)], 1);
    const int n = p / top, t = p % top;
    tok_of[r] = n;
    pair_of[r] = p;
    part_of[r] = t * n_tokens + n;
    weight_of[r] = weights[p];
  }
}

SYN_EXPORT int syn_route_sort(const int* ids, const float* weights, int* seg_start, int* tok_of, int* pair_of,
                              int* part_of, float* weight_of, int n_tokens, int top, int E, hipStream_t stream) {
  SYN_CHECK(n_tokens > 0 && top > 0, "route_sort: empty input");
  SYN_CHECK(E > 0 && E <= ROUTE_MAX_EXPERTS, "route_sort: %d experts (at most %d)", E, ROUTE_MAX_EXPERTS);
  SYN_CHECK((long)n_tokens * top < (1L << 30), "route_sort: %d tokens x %d", n_tokens, top);
  const int P = n_tokens * top, groups = min((P + SORT_PAIRS - 1) / SORT_PAIRS, SORT_GROUPS), share = (P + groups - 1) / groups;
  route_sort_kernel<<<groups, 1024, 0, stream>>>(ids, weights, seg_start, tok_of, pair_of, part_of, weight_of, n_tokens, top, E, share);
  SYN_LAUNCH_CHECK("route_sort");
  return 0;
}
