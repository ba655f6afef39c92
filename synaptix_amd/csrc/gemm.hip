// out[M, N] = x[M, K] . W[N, K]^T with 32-bit accumulation (both operands K-contiguous).
//
//   gemm_simt      any shape and type; plain FMA: what the MFMA kernels refuse (K not a multiple of 8, or of 4 in 32 bits;
//                  unaligned rows).
//   gemm_f32       32-bit, K a multiple of 4: gemm_f32.hip.
//   gemm_skinny    bf16, M == 1: the weight matrix is streamed once from HBM through
//                  v_mfma_f32_16x16x32_bf16; the waves of a workgroup split K and sum in LDS
//                  (also over paired gate/up rows, with the gated activation as the epilogue).
//   gemm_packed    bf16, M <= 16 (used up to 8): the same over a copy of W kept in the order of the MFMA
//                  fragments, so that every load of a wave is 1 KB of consecutive bytes.
//   gemm_stream    bf16, M > 64 (gated 16), K a multiple of 64: tiles of 256 x 256 down to 64 x 128, loads straight into LDS, one
//                  stream of k-steps over all tiles of a workgroup.
//   gemm_direct    bf16, up to 64 rows, and up to 256 where its tiles fill the compute units and go round once (large weights, or W in
//                  plain rows): 32 to 256 rows of x, 64 to 128 rows of W, 64 to 256 deep, straight into LDS: the rows of W arrive as whole
//                  256-byte pieces, which streams them faster than loading MFMA fragments (64 bytes a row) straight
//                  from memory.
//   gemm_tiled     bf16, any K that is a multiple of 8: the tiles pass through registers on their way to LDS.
//                  The last three: K may be cut into slices whose partial sums the reader adds; with paired rows W holds
//                  those of a gate and of an up projection in turns of 16 and the kernel stores act(gate) * up,
//                  half as wide, without the two products ever being stored.
//
// Reference counterparts: crates/synaptix-kernels-cuda/src/best_cu/gemm/gemm_bf16.cu (TN family,
// mma.sync m16n8k16), best_cu/gemv/mma_gemv.cu:19-133 (M == 1), best_cu/gemm/gemm_f32.cu (SIMT).
// The tilings here are made for 64-lane waves and MFMA operand layouts, not translated.
#include <algorithm>
#include <type_traits>

#include "common.h"

// What a kernel does with its 32-bit sums: store them as float or as bf16, behind `point` of point_activation if one is
// asked for, or (the kernels over paired gate/up rows) store act(gate) * up as bf16 with the activation `act` of
// gate_activation.
struct Epilogue {
  int out_is_f32;
  int act;
  float limit;      // the bound of an activation that has one (gated, csrc/common.h)
  int point;        // SYN_POINT_NONE, or what a plain product's sums pass before they are stored
  int add = 0;      // float results of the streamed tiles: added to what the output holds
};

// ------------------------------------------------------------------ SIMT, any type
#define SIMT_BM 64
#define SIMT_BN 64
#define SIMT_BK 16

template <typename TIn, typename TOut>
__global__ void __launch_bounds__(256)
gemm_simt_kernel(const TIn* __restrict__ x, const TIn* __restrict__ w, TOut* __restrict__ out, int M, int N, int K,
                 int point) {
  __shared__ float xs[SIMT_BK][SIMT_BM + 1];
  __shared__ float ws[SIMT_BK][SIMT_BN + 1];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * SIMT_BM, n0 = blockIdx.x * SIMT_BN;
  const int tm = (tid / 16) * 4, tn = (tid % 16) * 4;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += SIMT_BK) {
    // 64 rows x 16 k for each operand: 1024 values, 4 a thread
    for (int e = tid; e < SIMT_BM * SIMT_BK; e += 256) {
      const int r = e / SIMT_BK, kk = e % SIMT_BK;
      const int gm = m0 + r, gn = n0 + r, gk = k0 + kk;
      xs[kk][r] = (gm < M && gk < K) ? to_f32<TIn>(x[(size_t)gm * K + gk]) : 0.f;
      ws[kk][r] = (gn < N && gk < K) ? to_f32<TIn>(w[(size_t)gn * K + gk]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < SIMT_BK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[kk][tm + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[kk][tn + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gm = m0 + tm + i, gn = n0 + tn + j;
      if (gm < M && gn < N) out[(size_t)gm * N + gn] = from_f32<TOut>(point_activation(point, acc[i][j]));
    }
}

// ------------------------------------------------------------------ skinny, bf16, one row of x (up to 16)
// MFMA 16x16x32: A = x rows (m), B = W rows (n), D[m = 4*(lane/16)+j][n = lane%16].
// Both operands: lane holds row lane%16, k = 8*(lane/16) .. +8, one 16-byte load.
// A workgroup owns TILES * 16 rows of W, 16 for each group of KWAVES waves; the waves of a group take
// k-chunks of 32 round-robin, so that at any moment the group reads KWAVES*64 contiguous bytes of each
// row, and their partial tiles are summed in LDS in a fixed order.  PAIRED (TILES == 2): the first 16
// rows are gate rows, the second the up rows of the same outputs, and silu(gate) * up is stored.
template <int TILES, int KWAVES, int U, bool PAIRED>
__global__ void __launch_bounds__(TILES * KWAVES * SYN_WAVE)
gemm_skinny_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, void* __restrict__ out, Epilogue ep,
                   int M, int N, int K) {
  static_assert(!PAIRED || TILES == 2, "a pair is two tiles");
  constexpr int WAVES = TILES * KWAVES;
  __shared__ float part[WAVES][4][64];
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  const int tile = wave / KWAVES, kw = wave % KWAVES;
  const int r16 = lane % 16, kq = (lane / 16) * 8;
  const int n0 = (blockIdx.x * TILES + tile) * 16;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};

  // Rows of W beyond N are read from the last valid row (their results are never stored); rows of x
  // beyond M are not loaded at all: the fewer lanes a load of x has, the less it costs.
  const bf16* wrow = w + (size_t)min(n0 + r16, N - 1) * K + kq;
  const bool xok = r16 < M;
  const bf16* xrow = x + (size_t)min(r16, M - 1) * K + kq;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};

  // U chunks of 32 at a time: all loads of a group are issued before the first product needs them,
  // so that a wave keeps U KiB of the weight stream in flight
  constexpr int GROUP = 32 * U;
  const int k_full = K / (KWAVES * GROUP) * (KWAVES * GROUP);
  for (int k0 = kw * GROUP; k0 < k_full; k0 += KWAVES * GROUP) {
    bf16x8 bw[U], ax[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bw[u] = __builtin_nontemporal_load((const bf16x8*)(wrow + k0 + u * 32));
      ax[u] = xok ? *(const bf16x8*)(xrow + k0 + u * 32) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[u], bw[u], acc, 0, 0, 0);
  }
  // what is left of K, chunk by chunk; K is a multiple of 8, so a lane's 8 elements lie inside or
  // outside as a whole
  for (int k0 = k_full + kw * 32; k0 < K; k0 += KWAVES * 32) {
    const bool kin = k0 + kq < K;
    const bf16x8 ax = (kin && xok) ? *(const bf16x8*)(xrow + k0) : zero;
    const bf16x8 bw = kin ? *(const bf16x8*)(wrow + k0) : zero;
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax, bw, acc, 0, 0, 0);
  }

#pragma unroll
  for (int j = 0; j < 4; ++j) part[wave][j][lane] = acc[j];
  __syncthreads();
  auto summed = [&](int t, int j, int ln) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < KWAVES; ++q) s += part[t * KWAVES + q][j][ln];
    return s;
  };
  if constexpr (PAIRED) {
    for (int idx = threadIdx.x; idx < 4 * 64; idx += WAVES * SYN_WAVE) {
      const int j = idx / 64, ln = idx % 64;
      const int m = 4 * (ln / 16) + j, col = (int)blockIdx.x * 16 + ln % 16;  // N / 2 outputs, 16 a workgroup
      if (m < M && 2 * col < N) {
        const float g = summed(0, j, ln), up = summed(1, j, ln);
        ((bf16*)out)[(size_t)m * (N / 2) + col] = (bf16)gated(ep.act, g, up, ep.limit);
      }
    }
  } else {
    for (int idx = threadIdx.x; idx < TILES * 4 * 64; idx += WAVES * SYN_WAVE) {
      const int t = idx / 256, j = (idx / 64) % 4, ln = idx % 64;
      const int m = 4 * (ln / 16) + j, n = (blockIdx.x * TILES + t) * 16 + ln % 16;
      if (m < M && n < N) {
        const float v = point_activation(ep.point, summed(t, j, ln));
        if (ep.out_is_f32)
          ((float*)out)[(size_t)m * N + n] = v;
        else
          ((bf16*)out)[(size_t)m * N + n] = (bf16)v;
      }
    }
  }
}

template <int TILES, int KWAVES, int U, bool PAIRED = false>
static void launch_skinny(const bf16* x, const bf16* w, void* out, Epilogue ep, int M, int N, int K,
                          hipStream_t stream) {
  const int rows = TILES * 16;
  gemm_skinny_kernel<TILES, KWAVES, U, PAIRED>
      <<<(N + rows - 1) / rows, TILES * KWAVES * SYN_WAVE, 0, stream>>>(x, w, out, ep, M, N, K);
}

// ------------------------------------------------------------------ a norm between two products for few rows
// RMSNorm between two products for few rows of x needs every element of a row, which no workgroup of the product
// before it holds; as a kernel of its own it moves a few KB and costs a launch.  The products over packed
// weights therefore carry it between them in two halves:
//   * the product BEFORE the norm (resid != null; one slice of K, float sums) adds its sums into the float residual
//     rows, stores xs[m, n] = bf16((gain_offset + gain[n]) * resid[m, n]) (the norm's input with the gain, without
//     the row's factor) and, for each group of 16 columns, ss_out[m, group] = the sum of resid[m, n]^2 over them;
//   * the product AFTER the norm (ss != null) takes xs as its x and multiplies its finished sums of row m by
//     rsqrt(sum over groups of ss[m, :] / dim + eps): the product is linear in x, so the row's factor can wait.
// A row's statistic is added up in a fixed order (groups in turn over the lanes, then the wave's tree).
struct RowNorm {
  const float* ss;    // [M, ss_groups] of the product before, or null
  int ss_groups;
  float inv_dim;      // 1 / width of the normed rows
  float eps;
  float* resid;       // [M, N] float, or null
  bf16* xs;           // [M, N]
  float* ss_out;      // [M, N / 16]
  const void* gain;   // [N] bf16 or float
  int gain_is_f32;
  float gain_offset;
  const float* add_rows;   // [M, N] or null: what else the residual rows get (parts.linear.InjectedDelta)
  const float* add_vec;    // [N] or null: the same for every row
};

// inv[m] for the rows of x into LDS (16 floats): wave w takes rows w and w + n_waves (up to 16 rows, 8 waves or more).
// The statistic's first 256 groups a row are asked for before the product's loop (row_stat_load) and added up behind
// it (row_stat_finish), so that their way from memory is not the tail of the workgroup.
struct RowStat {
  float v[2][4];
};
__device__ __forceinline__ void row_stat_load(const RowNorm& rn, int M, int wave, int n_waves, int lane, RowStat& st) {
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int m = wave + r * n_waves;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = lane + SYN_WAVE * i;
      st.v[r][i] = (rn.ss && m < M && t < rn.ss_groups) ? rn.ss[(size_t)m * rn.ss_groups + t] : 0.f;
    }
  }
}
__device__ __forceinline__ void row_stat_finish(const RowNorm& rn, int M, int wave, int n_waves, int lane, const RowStat& st,
                                                float* inv) {
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int m = wave + r * n_waves;
    if (m >= M) break;   // the same for the whole wave
    float s = (st.v[r][0] + st.v[r][1]) + (st.v[r][2] + st.v[r][3]);
    for (int t = lane + 4 * SYN_WAVE; t < rn.ss_groups; t += SYN_WAVE) s += rn.ss[(size_t)m * rn.ss_groups + t];
    s = wave_sum(s);
    if (lane == 0) inv[m] = rsqrtf(s * rn.inv_dim + rn.eps);
  }
}

// the epilogue of the product before the norm for output (m, n) with its finished sum v; all 16 lanes of a
// group of columns call it together (rows beyond M with in == false); r0 and g: resid[m, n] and the gain of
// column n, asked for before the product's loop
__device__ __forceinline__ void resid_norm_store(const RowNorm& rn, bool in, int m, int n, int N, float v, float r0, float g) {
  float r = 0.f;
  if (in) {
    const size_t at = (size_t)m * N + n;
    r = r0 + v;
    rn.resid[at] = r;
    rn.xs[at] = (bf16)(g * r);
  }
  float q = r * r;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) q += __shfl_xor(q, off, SYN_WAVE);
  if (in && (n & 15) == 0) rn.ss_out[(size_t)m * (N / 16) + n / 16] = q;
}

// what the sums of the products for few rows may pass before they are stored: the points of every product, and a soft cap
__device__ __forceinline__ float packed_point(const Epilogue& ep, float v) {
  return ep.point == SYN_POINT_SOFTCAP ? soft_cap(v, ep.limit) : point_activation(ep.point, v);
}

// ------------------------------------------------------------------ few rows of x, W in fragment order
// The same scheme as gemm_skinny (up to 16 rows of x, K split over the waves of a group, partial
// tiles summed in LDS in a fixed order) over a copy of W that is kept in the order of the MFMA
// fragments: wp[N / 16][K / 32][64 lanes][8], lane = 16 * (k % 32 / 8) + n % 16.  A wave's load of a
// fragment is then 1 KB of consecutive bytes, and the fragments of a group of rows follow each other
// along K: the weight stream is read as a kernel that does nothing else reads it (measured 6.2 to
// 6.7 TB/s on the wide products, against 4.5 to 5.3 from rows of W).  The fragments of x come from
// memory for every wave (x stays in the caches); that costs as many requests as W from 16 rows on,
// so the callers use this kernel up to 8 rows.  Wave kw of a group takes the k-steps kw * U .. + U,
// then those KWAVES * U further on.
//
// The rows of x as these kernels load them: lane r16 + 16 q has k-values 8 q .. + 8 of row r16.  EIGHT: of up to eight rows, lanes
// r16 < 8 those of one k-step and lanes r16 >= 8 those of the next, so that a load asks for whole lines of 128 bytes.  A product with
// W's fragment of the first k-step then leaves its sums in rows 0 to 7 and one with that of the next in rows 8 to 15; what stands
// in the other rows mixes the two and is never read.  For plain products of 5 to 8 rows: 8 rows through 12,288 x 4,096 17.8 -> 16.8 us,
// 10,304 x 4,096 16.9 -> 15.9, 5,120 x 25,600 62.8 -> 58.1, 4,096 x 12,288 18.7 -> 18.2, 4,096 x 4,096 7.55, 7.52; 5 rows 16.7, 16.5,
// 16.0, 15.1, 57.7, 56.1, 17.8, 17.9, 7.5, 7.5.  Fewer rows cost few requests either way and lost up to 1.5 us; gated products,
// whose x serves two groups of rows of W, gained nothing (33.2, 33.5).
template <bool EIGHT>
struct XRows {
  const bf16* row;
  bool ok;
  int behind;
  __device__ __forceinline__ XRows(const bf16* x, int M, int K, int r16, int kq) {
    const int r = EIGHT ? r16 % 8 : r16;
    behind = EIGHT ? r16 / 8 : 0;
    ok = r < M;
    row = x + (size_t)min(r, M - 1) * K + behind * 32 + kq;
  }
  __device__ __forceinline__ bf16x8 load(int ks, int ks_end) const {
    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    return ok && ks + behind < ks_end ? *(const bf16x8*)(row + ks * 32) : zero;
  }
};

template <int TILES, int KWAVES, int U, bool PAIRED, bool EIGHT>
__global__ void __launch_bounds__(TILES * KWAVES * SYN_WAVE)
gemm_packed_kernel(const bf16* __restrict__ x, const bf16* __restrict__ wp, void* __restrict__ out, Epilogue ep,
                   int M, int N, int K, int ks_slice, RowNorm rn) {
  static_assert(!PAIRED || TILES == 2, "a pair is two tiles");
  constexpr int WAVES = TILES * KWAVES;
  __shared__ float part[WAVES][4][64];
  __shared__ float inv[16];
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  const int tile = wave / KWAVES, kw = wave % KWAVES;
  const int r16 = lane % 16, kq = (lane / 16) * 8;
  const int nt = (int)blockIdx.x * TILES + tile, n_tiles = N / 16;   // 16 rows of W
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const int nks = K / 32;
  const bool tile_in = nt < n_tiles;   // the last workgroup may hold a group beyond the end
  const bf16* wt = wp + ((size_t)min(nt, n_tiles - 1) * nks * 64 + lane) * 8;
  const XRows<EIGHT> xr(x, M, K, r16, kq);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc_odd = {0.f, 0.f, 0.f, 0.f};
  // what the epilogue needs of a norm's halves is asked for now, not behind the loop
  RowStat stat;
  if (rn.ss) row_stat_load(rn, M, wave, WAVES, lane, stat);
  float r0 = 0.f, g0 = 0.f;
  static_assert(TILES * 256 <= WAVES * SYN_WAVE, "every thread stores at most one output");
  if (!PAIRED && rn.resid && threadIdx.x < TILES * 256) {
    const int t = threadIdx.x / 256, j = (threadIdx.x / 64) % 4, ln = threadIdx.x % 64;
    const int m = 4 * (ln / 16) + j, n = ((int)blockIdx.x * TILES + t) * 16 + ln % 16;
    if (m < M && n < N) {
      r0 = rn.resid[(size_t)m * N + n], g0 = load_gain(rn.gain, rn.gain_is_f32, n, rn.gain_offset);
      if (rn.add_rows) r0 += rn.add_rows[(size_t)m * N + n];
      if (rn.add_vec) r0 += rn.add_vec[n];
    }
  }
  // blockIdx.y = which slice of K (ks_slice k-steps of 32) this workgroup sums; its output is slice blockIdx.y
  // of a float [slices, M, N] that the reader adds up (a product with few rows of W gets more workgroups so)
  const int ks_begin = (int)blockIdx.y * ks_slice, ks_end = min(nks, ks_begin + ks_slice);
  if (tile_in) {
    for (int ks0 = ks_begin + kw * U; ks0 < ks_end; ks0 += KWAVES * U) {
      bf16x8 bw[U], ax[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = ks0 + u < ks_end;
        bw[u] = in ? __builtin_nontemporal_load((const bf16x8*)(wt + (size_t)(ks0 + u) * 512)) : zero;
        if (!EIGHT || u % 2 == 0) ax[u] = xr.load(ks0 + u, ks_end);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (EIGHT && u % 2) acc_odd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[u - 1], bw[u], acc_odd, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[u], bw[u], acc, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) part[wave][j][lane] = EIGHT && lane >= 32 ? acc_odd[j] : acc[j];
  if (rn.ss) row_stat_finish(rn, M, wave, WAVES, lane, stat, inv);
  __syncthreads();
  auto summed = [&](int t, int j, int ln) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < KWAVES; ++q) s += EIGHT ? part[t * KWAVES + q][j][ln % 32] + part[t * KWAVES + q][j][ln % 32 + 32] : part[t * KWAVES + q][j][ln];
    return s;
  };
  if constexpr (PAIRED) {
    for (int idx = threadIdx.x; idx < 4 * 64; idx += WAVES * SYN_WAVE) {
      const int j = idx / 64, ln = idx % 64;
      const int m = 4 * (ln / 16) + j, col = (int)blockIdx.x * 16 + ln % 16;  // N / 2 outputs, 16 a workgroup
      if (m < M && 2 * col < N) {
        const float f = rn.ss ? inv[m] : 1.f;
        const float g = summed(0, j, ln) * f, up = summed(1, j, ln) * f;
        ((bf16*)out)[(size_t)m * (N / 2) + col] = (bf16)gated(ep.act, g, up, ep.limit);
      }
    }
  } else {
    for (int idx = threadIdx.x; idx < TILES * 4 * 64; idx += WAVES * SYN_WAVE) {
      const int t = idx / 256, j = (idx / 64) % 4, ln = idx % 64;
      const int m = 4 * (ln / 16) + j, n = ((int)blockIdx.x * TILES + t) * 16 + ln % 16;
      const bool in = m < M && n < N;
      float v = summed(t, j, ln);
      if (rn.ss && in) v *= inv[m];
      if (rn.resid) {   // the same for the whole workgroup
        resid_norm_store(rn, in, m, n, N, v, r0, g0);
      } else if (in) {
        v = packed_point(ep, v);
        if (ep.out_is_f32)
          ((float*)out)[((size_t)blockIdx.y * M + m) * N + n] = v;
        else
          ((bf16*)out)[(size_t)m * N + n] = (bf16)v;
      }
    }
  }
}

template <int TILES, int KWAVES, int U, bool PAIRED, bool EIGHT>
static void launch_packed_as(const bf16* x, const bf16* wp, void* out, Epilogue ep, int M, int N, int K,
                          hipStream_t stream, int slices, const RowNorm& rn) {
  const int rows = TILES * 16;
  const int ks_slice = (K / 32 + slices - 1) / slices;
  gemm_packed_kernel<TILES, KWAVES, U, PAIRED, EIGHT>
      <<<dim3((N + rows - 1) / rows, slices), TILES * KWAVES * SYN_WAVE, 0, stream>>>(x, wp, out, ep, M, N, K, ks_slice, rn);
}
template <int TILES, int KWAVES, int U, bool PAIRED = false>
static void launch_packed(const bf16* x, const bf16* wp, void* out, Epilogue ep, int M, int N, int K,
                          hipStream_t stream, int slices, const RowNorm& rn) {
  if constexpr (!PAIRED) {
    if (M >= 5 && M <= 8) return launch_packed_as<TILES, KWAVES, U, PAIRED, true>(x, wp, out, ep, M, N, K, stream, slices, rn);
  }
  launch_packed_as<TILES, KWAVES, U, PAIRED, false>(x, wp, out, ep, M, N, K, stream, slices, rn);
}


// The same with two adjacent groups of 16 rows of W for every wave (for PAIRED: the gate rows and the up rows of
// the same 16 outputs): a fragment of x is loaded once for two products, a third fewer loads at 8 rows of x.
template <int KWAVES, int U, bool PAIRED>
__global__ void __launch_bounds__(KWAVES * SYN_WAVE)
gemm_packed2_kernel(const bf16* __restrict__ x, const bf16* __restrict__ wp, void* __restrict__ out, Epilogue ep,
                    int M, int N, int K, int ks_slice, RowNorm rn) {
  __shared__ float part[KWAVES][2][4][64];
  __shared__ float inv[16];
  const int kw = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  const int r16 = lane % 16, kq = (lane / 16) * 8;
  const int nt = (int)blockIdx.x * 2, n_tiles = N / 16;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const int nks = K / 32;
  const bool second = nt + 1 < n_tiles;   // an odd number of groups leaves the last workgroup one
  const bf16* wt0 = wp + ((size_t)nt * nks * 64 + lane) * 8;
  const bf16* wt1 = wp + ((size_t)min(nt + 1, n_tiles - 1) * nks * 64 + lane) * 8;
  const bool xok = r16 < M;
  const bf16* xrow = x + (size_t)min(r16, M - 1) * K + kq;
  f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  RowStat stat;
  if (rn.ss) row_stat_load(rn, M, kw, KWAVES, lane, stat);
  const int ks_begin = (int)blockIdx.y * ks_slice, ks_end = min(nks, ks_begin + ks_slice);
  for (int ks0 = ks_begin + kw * U; ks0 < ks_end; ks0 += KWAVES * U) {
    bf16x8 b0[U], b1[U], ax[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = ks0 + u < ks_end;
      b0[u] = in ? __builtin_nontemporal_load((const bf16x8*)(wt0 + (size_t)(ks0 + u) * 512)) : zero;
      b1[u] = in ? __builtin_nontemporal_load((const bf16x8*)(wt1 + (size_t)(ks0 + u) * 512)) : zero;
      ax[u] = (in && xok) ? *(const bf16x8*)(xrow + (ks0 + u) * 32) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[u], b0[u], acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax[u], b1[u], acc1, 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) part[kw][0][j][lane] = acc0[j], part[kw][1][j][lane] = acc1[j];
  if (rn.ss) row_stat_finish(rn, M, kw, KWAVES, lane, stat, inv);
  __syncthreads();
  auto summed = [&](int t, int j, int ln) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < KWAVES; ++q) s += part[q][t][j][ln];
    return s;
  };
  if constexpr (PAIRED) {
    for (int idx = threadIdx.x; idx < 4 * 64; idx += KWAVES * SYN_WAVE) {
      const int j = idx / 64, ln = idx % 64;
      const int m = 4 * (ln / 16) + j, col = (int)blockIdx.x * 16 + ln % 16;  // N / 2 outputs, 16 a workgroup
      if (m < M && 2 * col < N) {
        const float f = rn.ss ? inv[m] : 1.f;
        ((bf16*)out)[(size_t)m * (N / 2) + col] = (bf16)gated(ep.act, summed(0, j, ln) * f, summed(1, j, ln) * f, ep.limit);
      }
    }
  } else {
    for (int idx = threadIdx.x; idx < 2 * 4 * 64; idx += KWAVES * SYN_WAVE) {
      const int t = idx / 256, j = (idx / 64) % 4, ln = idx % 64;
      const int m = 4 * (ln / 16) + j, n = (nt + t) * 16 + ln % 16;
      if (m < M && n < N && (t == 0 || second)) {
        float v = summed(t, j, ln);
        if (rn.ss) v *= inv[m];
        v = packed_point(ep, v);
        if (ep.out_is_f32) ((float*)out)[((size_t)blockIdx.y * M + m) * N + n] = v;
        else ((bf16*)out)[(size_t)m * N + n] = (bf16)v;
      }
    }
  }
}

template <int KWAVES, int U, bool PAIRED = false>
static void launch_packed2(const bf16* x, const bf16* wp, void* out, Epilogue ep, int M, int N, int K,
                           hipStream_t stream, int slices, const RowNorm& rn) {
  const int ks_slice = (K / 32 + slices - 1) / slices;
  gemm_packed2_kernel<KWAVES, U, PAIRED>
      <<<dim3((N + 31) / 32, slices), KWAVES * SYN_WAVE, 0, stream>>>(x, wp, out, ep, M, N, K, ks_slice, rn);
}

// ------------------------------------------------------------------ shared by the tiled kernels
// Which tile: workgroup b runs on XCD b % 8, and each XCD has an L2 of its own.  Tiles are grouped
// into panels of PM x PN (m fastest); a panel goes to one XCD, so the workgroups that run there at
// the same time share rows of x and of W in its L2.  False for the launches that pad the last panels.
// With slices of K (blockIdx.y) the panels of slice s are handed out s * panels XCDs further on, so
// that a product of fewer than 8 panels still reaches every XCD.
__device__ __forceinline__ bool tile_of_workgroup(int M, int N, int BM, int BN, int& tm, int& tn) {
  const int tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
  const int PM = min(8, tiles_m), PN = 4;
  const int panels_m = (tiles_m + PM - 1) / PM, panels = panels_m * ((tiles_n + PN - 1) / PN);
  const int xcd = ((int)blockIdx.x + 8 - (int)((blockIdx.y * panels) % 8)) % 8, local = (int)blockIdx.x / 8;
  const int panel = (local / (PM * PN)) * 8 + xcd, in_panel = local % (PM * PN);
  tm = (panel % panels_m) * PM + in_panel % PM;
  tn = (panel / panels_m) * PN + in_panel / PM;
  return tm < tiles_m && tn < tiles_n;
}

static int tile_grid(int M, int N, int BM, int BN) {
  const int tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
  const int PM = tiles_m < 8 ? tiles_m : 8, PN = 4;
  const int panels = ((tiles_m + PM - 1) / PM) * ((tiles_n + PN - 1) / PN);
  return (panels + 7) / 8 * 8 * PM * PN;
}

// The accumulators of a wave (TM x TN tiles of MFMA 32x32: D[m = 8*(e/4) + 4*(lane/32) + e%4][n = lane%32])
// to memory.  mw, nw: the first row and column of the wave's part.  PAIRED: columns n % 32 < 16 are
// gate rows, the 16 after them the up rows of the same outputs (N is a multiple of 32 then, so a tile of
// 32 columns lies inside or outside as a whole).  Two tiles side by side are stored together: the lanes
// of the first kind take the first tile (their own gate, the partner's up), the others the second (the
// partner's gate, their own up), so that a store covers 32 consecutive outputs of a row (64 bytes, not
// twice 32).  A last tile without a neighbour is stored by the lanes of the first kind alone.
// QUICK: the gated activation as the streamed tiles apply it, so that a product's bits do not depend on which of the two it takes
// (W in plain rows or in fragment order).
template <bool QUICK>
__device__ __forceinline__ float gated_epilogue(const Epilogue& ep, float g, float up) {
  if constexpr (!QUICK) return gated(ep.act, g, up, ep.limit);
  if (ep.act == SYN_ACT_SILU) return gated_quick<SYN_ACT_SILU, false>(g, up, 0.f);
  if (ep.act == SYN_ACT_SWIGLU_LIMIT) return gated_quick<SYN_ACT_SWIGLU_LIMIT, false>(g, up, ep.limit);
  return gated_quick<SYN_ACT_GELU_TANH, false>(g, up, 0.f);
}
template <int TM, int TN, bool PAIRED, bool QUICK = false>
__device__ __forceinline__ void store_tiles(const f32x16 (&acc)[TM][TN], void* __restrict__ out, Epilogue ep,
                                            size_t slice, int M, int N, int mw, int nw, int lane) {
  if constexpr (PAIRED) {
    const bool first = lane % 32 < 16;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; j += 2)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = mw + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
          const float own0 = acc[i][j][e], other0 = __shfl_xor(own0, 16, SYN_WAVE);
          if (j + 1 < TN) {   // known once the loop is unrolled
            const float own1 = acc[i][j + 1 < TN ? j + 1 : j][e], other1 = __shfl_xor(own1, 16, SYN_WAVE);
            const float g = first ? own0 : other1, up = first ? other0 : own1;
            if (m < M && nw + (j + (first ? 0 : 1)) * 32 < N)
              ((bf16*)out)[(size_t)m * (N / 2) + (nw + j * 32) / 2 + lane % 32] = (bf16)gated_epilogue<QUICK>(ep, g, up);
          } else {
            if (m < M && nw + j * 32 < N && first)
              ((bf16*)out)[(size_t)m * (N / 2) + (nw + j * 32) / 2 + lane % 16] = (bf16)gated_epilogue<QUICK>(ep, own0, other0);
          }
        }
  } else {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = mw + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
          const int n = nw + j * 32 + lane % 32;
          if (m < M && n < N) {
            const float v = point_activation(ep.point, acc[i][j][e]);
            if (ep.out_is_f32)
              ((float*)out)[(slice * M + m) * N + n] = v;
            else
              ((bf16*)out)[(size_t)m * N + n] = (bf16)v;
          }
        }
  }
}

// ------------------------------------------------------------------ tiled, bf16
// Block tile BM (m) x BN (n) x BK (k); WM x WN waves, each (BM/WM) x (BN/WN) of MFMA 32x32x16 tiles.
// MFMA 32x32x16: A = x rows, B = W rows; lane holds row lane%32, k = 8*(lane/32) .. +8;
// D[m = 8*(j/4) + 4*(lane/32) + j%4][n = lane%32], j = 0..15.
// LDS tiles are double-buffered: while one k-tile is multiplied the next is on its way from memory
// into registers, and is stored into the other buffer before the barrier.
template <int BM, int BN, int BK, int WM, int WN, bool KTAIL, bool PAIRED>
__global__ void __launch_bounds__(64 * WM * WN)
gemm_tiled_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, void* __restrict__ out, Epilogue ep,
                  int M, int N, int K, int k_slice) {
  constexpr bool FEW = BM <= 64;                     // the variants for few rows of x: slices of K, absent rows
  constexpr int THREADS = 64 * WM * WN;              // WM x WN waves
  constexpr int LD = BK + 8;                         // padded row of the LDS tiles, in bf16 elements
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // 32x32 tiles a wave holds in m and n
  constexpr int CPR = BK / 8;                        // 16-byte chunks in a tile row
  constexpr int RPP = THREADS / CPR;                 // tile rows the workgroup moves in one pass
  constexpr int XL = BM / RPP, WL = BN / RPP;        // passes for x and for W
  static_assert(BM % RPP == 0 && BN % RPP == 0 && TM >= 1 && TN >= 1, "tile shape");
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];  // [2][(BM + BN) * LD]
  const int tid = threadIdx.x, wave = tid / SYN_WAVE, lane = tid % SYN_WAVE;
  const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
  int tm, tn;
  if (!tile_of_workgroup(M, N, BM, BN, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};

  // global -> LDS: thread t moves chunk t % CPR of rows t / CPR + RPP * i
  const int lrow = tid / CPR, lchunk = (tid % CPR) * 8;
  // rows of x beyond M are not fetched (their LDS rows hold zeros and their results are never
  // stored): with few rows this spares most of the traffic for x
  const bf16* xg[XL];
  const bf16* wg[WL];
  bool xin[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    xin[i] = !FEW || m0 + lrow + RPP * i < M;
    xg[i] = x + (size_t)min(m0 + lrow + RPP * i, M - 1) * K + lchunk;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) wg[i] = w + (size_t)min(n0 + lrow + RPP * i, N - 1) * K + lchunk;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // blockIdx.y = which slice of K (k_slice elements, a multiple of 128) this workgroup sums
  const int k_begin = FEW ? (int)blockIdx.y * k_slice : 0, k_end = FEW ? min(K, k_begin + k_slice) : K;
  const int nk = (k_end - k_begin + BK - 1) / BK;
  bf16x8 rx[XL], rw[WL];
  auto fetch = [&](int kt) {
    // K is a multiple of 8: a chunk lies inside or outside as a whole
    const int k = k_begin + kt * BK;
    const bool kin = !KTAIL || k + lchunk < k_end;
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      rx[i] = (kin && xin[i]) ? *(const bf16x8*)(xg[i] + k) : zero;
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) rw[i] = kin ? *(const bf16x8*)(wg[i] + k) : zero;
  };
  auto stash = [&](int buf) {
    bf16* xs = smem + buf * (BM + BN) * LD;
    bf16* ws = xs + BM * LD;
#pragma unroll
    for (int i = 0; i < XL; ++i) *(bf16x8*)(xs + (lrow + RPP * i) * LD + lchunk) = rx[i];
#pragma unroll
    for (int i = 0; i < WL; ++i) *(bf16x8*)(ws + (lrow + RPP * i) * LD + lchunk) = rw[i];
  };

  fetch(0);
  stash(0);
  __syncthreads();
  const int fr = lane % 32, fk = (lane / 32) * 8;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) fetch(kt + 1);
    const bf16* xs = smem + buf * (BM + BN) * LD;
    const bf16* ws = xs + BM * LD;
#pragma unroll
    for (int ks = 0; ks < BK; ks += 16) {
      bf16x8 a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = *(const bf16x8*)(xs + (wm + i * 32 + fr) * LD + ks + fk);
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = *(const bf16x8*)(ws + (wn + j * 32 + fr) * LD + ks + fk);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) stash(buf ^ 1);  // the other buffer was last read before the previous barrier
    __syncthreads();
  }

  store_tiles<TM, TN, PAIRED>(acc, out, ep, FEW ? blockIdx.y : 0, M, N, m0 + wm, n0 + wn, lane);
}

template <int BM, int BN, int BK, int WM, int WN, bool PAIRED = false>
static int launch_tiled(const bf16* x, const bf16* w, void* out, Epilogue ep, int M, int N, int K,
                        hipStream_t stream, int slices = 1) {
  SYN_CHECK(slices == 1 || BM <= 64, "gemm: slices of K only with the tiles for few rows");   // (gemm_tiled's own limit)
  const int k_slice = ((K + slices - 1) / slices + 127) / 128 * 128;  // the same cut as launch_direct makes
  const int grid = tile_grid(M, N, BM, BN);
  const size_t lds = (size_t)2 * (BM + BN) * (BK + 8) * sizeof(bf16);
  static OncePerDevice raised;
  if (lds > 65536) {
    const hipError_t e = once_per_device(raised, [&] {
      hipError_t r = hipFuncSetAttribute((const void*)gemm_tiled_kernel<BM, BN, BK, WM, WN, false, PAIRED>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (r == hipSuccess)
        r = hipFuncSetAttribute((const void*)gemm_tiled_kernel<BM, BN, BK, WM, WN, true, PAIRED>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      return r;
    });
    SYN_CHECK(e == hipSuccess, "gemm: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
  }
  // whole k-tiles only, and no slice that begins at or beyond the end of K: then no chunk needs a check
  if (K % BK == 0 && k_slice % BK == 0 && (long)(slices - 1) * k_slice < K)
    gemm_tiled_kernel<BM, BN, BK, WM, WN, false, PAIRED>
        <<<dim3(grid, slices), 64 * WM * WN, lds, stream>>>(x, w, out, ep, M, N, K, k_slice);
  else
    gemm_tiled_kernel<BM, BN, BK, WM, WN, true, PAIRED>
        <<<dim3(grid, slices), 64 * WM * WN, lds, stream>>>(x, w, out, ep, M, N, K, k_slice);
  return 0;
}

// ------------------------------------------------------------------ tiled, loads straight into LDS
// The same tiles with buffer_load_dwordx4 ... lds: a load writes its 16 bytes a lane into LDS without
// passing through registers, so a k-tile on its way costs no registers and no LDS store
// instructions, and the wait for it is the last thing before the barrier.  K (and every slice of
// it) must be a multiple of BK.  An instruction of a wave fills 1 KB of LDS in lane order: 8 rows of
// 64 k-values or 4 rows of 128, unpadded.  To keep the fragment reads free of bank conflicts all the
// same, slot s of row r holds the row's 16-byte chunk s ^ swizzle(r): the swizzle is applied to the
// global address of the lane that fills the slot, and again by the reader.  Measured 10 to 20 %
// faster than staging through registers for prompts, and for single tokens from 16 rows of x on.
template <int BK>
__device__ __forceinline__ int direct_swizzle(int row) {
  // BK = 64: a row is 128 bytes, two rows span the 64 banks; BK = 128: a row spans them all
  return BK == 64 ? (row >> 1) & 7 : row & (BK / 8 - 1);
}

// WP: w is the weight in fragment order (pack_weight: [N / 16][K / 32][64 lanes][8], N a multiple of 16).  A load of a
// wave then moves one fragment (16 rows x 32 k-values, 1 KB of consecutive bytes) into the slot that a load of
// plain rows fills, and a lane's fragment of an MFMA 32x32x16 lies in two of them: rows fr % 16 of fragment
// fr / 16, chunks 2 (ks % 2) + fh of k-fragment ks / 2; 16 lanes read 256 consecutive bytes, without a swizzle.
template <int BM, int BN, int BK, int WM, int WN, bool PAIRED, int STAGES, bool WP>
__global__ void __launch_bounds__(64 * WM * WN)
gemm_direct_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, void* __restrict__ out, Epilogue ep,
                   int M, int N, int K, int k_slice) {
  static_assert((BK == 64 || BK == 128 || BK == 256) && STAGES >= 2, "k-tiles of 64, 128 or 256 in two or more buffers");
  constexpr int WAVES = WM * WN;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int ROWS = BM + BN;
  constexpr int CPR = BK / 8;                    // 16-byte chunks in a row of a k-tile
  constexpr int RPI = 64 / CPR;                  // rows an instruction of a wave fills
  constexpr int PASSES = ROWS / (RPI * WAVES);   // instructions of a wave for one k-tile
  static_assert(ROWS % (RPI * WAVES) == 0 && TM >= 1 && TN >= 1, "tile shape");
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];  // [STAGES][ROWS][BK]
  const int tid = threadIdx.x, lane = tid % SYN_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / SYN_WAVE);   // scalar: LDS addresses of the loads stay scalar
  const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
  int tm, tn;
  if (!tile_of_workgroup(M, N, BM, BN, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN;
  // blockIdx.y = which slice of K (k_slice elements, a multiple of BK) this workgroup sums
  const int k_begin = (int)blockIdx.y * k_slice, k_end = min(K, k_begin + k_slice);
  const int nk = max(0, (k_end - k_begin) / BK);

  // the descriptors begin at the tile's first rows, so a lane's offset stays below 2^32 for any M and N,
  // and end with the last row of x and of W: a lane whose row lies beyond reads nothing from memory
  // (its LDS slot gets zeros, and its results are never stored), which with few rows of x spares
  // most of the requests for x.
  // pass p: the wave fills tile rows (p * WAVES + wave) * RPI .. + RPI (x rows first, then W rows)
  static_assert(BM % (RPI * WAVES) == 0, "a pass lies in x or in W as a whole, for all waves alike");
  const size_t row_bytes = (size_t)K * sizeof(bf16);
  const BufferView vx = buffer_view(x + (size_t)m0 * K, (size_t)(M - m0) * row_bytes);
  // (in fragment order 16 rows of W are K / 32 fragments of 1 KB one after another: as many bytes as 16 plain rows)
  const BufferView vw = buffer_view(w + (size_t)n0 * K, (size_t)(N - n0) * row_bytes);
  constexpr int KF = BK / 32;                    // fragments of a k-tile along K
  unsigned src[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int row0 = (p * WAVES + wave) * RPI, row = row0 + lane / CPR;
    const int chunk = (lane % CPR) ^ direct_swizzle<BK>(row);
    if (WP && row0 >= BM) {
      const int slot = (row0 - BM) / RPI;        // which fragment of the tile: 16 rows slot / KF, k-fragment slot % KF
      src[p] = (unsigned)((size_t)(slot / KF) * 16 * row_bytes + (size_t)(slot % KF) * 1024 + lane * 16);
    } else {
      const int in_tile = row0 < BM ? row : row - BM;
      src[p] = (unsigned)((size_t)in_tile * row_bytes + chunk * 16);
    }
  }
  auto fetch = [&](int kt, int buf) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      bf16* dst = smem + (size_t)buf * ROWS * BK + (size_t)(p * WAVES + wave) * RPI * BK;  // the same for all lanes
      // every wave fills rows of x in the first passes and rows of W in the others; this kernel runs where a
      // row of W has one reader (up to 64 rows of x) or at most four: its loads are marked non-temporal
      if (p * WAVES * RPI < BM)
        buffer_to_lds16(vx, dst, src[p], (k_begin + kt * BK) * (int)sizeof(bf16));
      else
        buffer_to_lds16<true>(vw, dst, src[p], (k_begin + kt * BK) * (int)sizeof(bf16) * (WP ? 16 : 1));
    }
  };
  // Tile kt lies in buffer kt % STAGES; while it is multiplied the STAGES - 1 tiles after it are on their
  // way.  Before the barrier that ends a tile a wave waits until its own loads of the next tile have
  // written LDS (all but the (STAGES - 2) * PASSES youngest have then) and its fragment reads have
  // returned.  The barrier carries no fence: a fence would wait for every load on its way.
  constexpr int YOUNGER = (STAGES - 2) * PASSES;
  auto next_landed = [](bool full_pipeline) {
    if (full_pipeline) __builtin_amdgcn_s_waitcnt(0x0070 | (YOUNGER & 15) | ((YOUNGER >> 4) << 14));
    else __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int fr = lane % 32, fh = lane / 32;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < nk) fetch(t, t);  // a slice beyond the end of K stores zeros
  next_landed(nk >= STAGES - 1);
  __builtin_amdgcn_s_barrier();
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt % STAGES;
    const bool more = kt + STAGES - 1 < nk;
    if (more) fetch(kt + STAGES - 1, (kt + STAGES - 1) % STAGES);  // that buffer was last read before the previous barrier
    const bf16* xs = smem + (size_t)buf * ROWS * BK;
    const bf16* ws = xs + BM * BK;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      bf16x8 a[TM], b[TN];
      const int c = 2 * ks + fh;  // the 16-byte chunk of a row that this lane multiplies
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm + i * 32 + fr;
        a[i] = *(const bf16x8*)(xs + row * BK + (c ^ direct_swizzle<BK>(row)) * 8);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn + j * 32 + fr;
        if constexpr (WP)
          b[j] = *(const bf16x8*)(ws + ((row / 16) * KF + ks / 2) * 512 + ((2 * (ks % 2) + fh) * 16 + row % 16) * 8);
        else
          b[j] = *(const bf16x8*)(ws + row * BK + (c ^ direct_swizzle<BK>(row + BM)) * 8);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    next_landed(more);
    __builtin_amdgcn_s_barrier();
  }
  store_tiles<TM, TN, PAIRED, true>(acc, out, ep, blockIdx.y, M, N, m0 + wm, n0 + wn, lane);
}

// A weight [N, K] as a product is handed it: plain rows, or in fragment order (pack_weight)
struct Weight {
  const bf16* p;
  bool packed;
};

// slices > 1 only with a float output [slices, M, N]; K must be a multiple of BK
template <int BM, int BN, int BK, int WM, int WN, bool PAIRED = false, int STAGES = 3>
static int launch_direct(const bf16* x, Weight w, void* out, Epilogue ep, int M, int N, int K,
                         hipStream_t stream, int slices = 1) {
  SYN_CHECK(K % BK == 0, "gemm: K = %d is no multiple of the k-tile %d", K, BK);
  const int step = BK > 128 ? BK : 128;
  const int k_slice = ((K + slices - 1) / slices + step - 1) / step * step;  // a multiple of BK
  const size_t lds = (size_t)STAGES * (BM + BN) * BK * sizeof(bf16);
  static OncePerDevice raised;
  if (lds > 65536) {
    const hipError_t e = once_per_device(raised, [&] {
      hipError_t r = hipFuncSetAttribute((const void*)gemm_direct_kernel<BM, BN, BK, WM, WN, PAIRED, STAGES, false>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (r == hipSuccess)
        r = hipFuncSetAttribute((const void*)gemm_direct_kernel<BM, BN, BK, WM, WN, PAIRED, STAGES, true>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      return r;
    });
    SYN_CHECK(e == hipSuccess, "gemm: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
  }
  const dim3 grid(tile_grid(M, N, BM, BN), slices);
  if (w.packed)
    gemm_direct_kernel<BM, BN, BK, WM, WN, PAIRED, STAGES, true><<<grid, 64 * WM * WN, lds, stream>>>(x, w.p, out, ep, M, N, K, k_slice);
  else
    gemm_direct_kernel<BM, BN, BK, WM, WN, PAIRED, STAGES, false><<<grid, 64 * WM * WN, lds, stream>>>(x, w.p, out, ep, M, N, K, k_slice);
  return 0;
}

// ------------------------------------------------------------------ 9 to 128 rows, W in fragment order: operands straight to registers
// (The rules take it up to 64 rows, gated 48; `rows` asks for it up to 128.)
// What bounds it: what a compute unit brings in, W and x together (13 to 15 bytes a clock), and W's stream from memory, of which a unit
// has to keep some 64 KB under way.  Through a ring of LDS buffers W shares the room with x (36 KB of it under way beside 96 rows
// of x), and every k-tile ends in a barrier.  Here the four waves of a workgroup
// (one a SIMD, all 512 registers) split K, and each takes all rows of x and all 16 NF rows of W of the workgroup: a fragment of
// either is loaded once a workgroup, straight into the registers of the one wave that multiplies it, S steps of 32 k-values ahead;
// no barrier and no LDS until the waves' sums are added at the end, in the order of the waves.  x comes from the L2s, as many
// bytes as W with 16 NF rows of it.
// W: a step's fragment is 1 KB of consecutive bytes; x: 16 rows of 64 bytes, the two steps of a 128-byte line asked for together.
// A wave takes every fourth pair of steps.  Rows of x beyond M, rows of W beyond N and steps beyond the slice lie behind the views'
// ends: zeros without traffic.  D[n = 4 (lane / 16) + e][m = lane % 16] of fragments (n, m).
template <int NF, int FM, int S, bool PAIRED>
__global__ void __launch_bounds__(256, 1)
gemm_rows_kernel(const bf16* __restrict__ x, const bf16* __restrict__ wp, void* __restrict__ out, Epilogue ep, int M, int N, int K,
                 int k_slice) {
  static_assert(NF % 2 == 0 && S % 2 == 0, "fragments of W in pairs (gate and up), steps in pairs (a line of x)");
  constexpr int FRAGS = NF * FM;
  static_assert(4 * FRAGS * SYN_WAVE * 16 <= 160 * 1024, "the waves' sums in LDS");
  // (256 vector registers beside the 256 of the sums.  With more, operands move between the two files next to the matrix
  // instructions, which the compiler does not know for what they are: 288 gave wrong results)
  static_assert(S * (NF + FM) * 4 <= 224 && FRAGS * 4 <= 256, "operands and sums in the registers of one wave a SIMD");
  extern __shared__ f32x4 part[];      // [4][FRAGS][64]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SYN_WAVE), lane = threadIdx.x % SYN_WAVE, r16 = lane % 16, g = lane / 16;
  const int n0 = (int)blockIdx.x * 16 * NF, k_begin = (int)blockIdx.y * k_slice;
  const int pairs = max(0, min(K - k_begin, k_slice)) / 64, steps = 2 * max(0, (pairs - wave + 3) / 4);
  const size_t row_bytes = (size_t)K * sizeof(bf16);
  const BufferView vw = buffer_view(wp + (size_t)n0 * K, (size_t)(N - n0) * row_bytes), vx = buffer_view(x, (size_t)M * row_bytes);
  const unsigned w_frag = (unsigned)(16 * row_bytes);
  const unsigned w_at = (unsigned)(k_begin / 32 + 2 * wave) * 1024 + lane * 16, x_at = (unsigned)(r16 * row_bytes) + (k_begin + 64 * wave + 8 * g) * 2;
  bf16x8 wf[S][NF], xf[S][FM];
  f32x4 acc[NF][FM];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // step s of this wave: pair wave + 4 (s / 2), half s % 2
  auto load_w = [&](int s, bf16x8 (&f)[NF]) {
    const unsigned at = w_at + (unsigned)((s / 2) * 8 + s % 2) * 1024;
#pragma unroll
    for (int i = 0; i < NF; ++i) f[i] = buffer_load16<true>(vw, s < steps ? at + i * w_frag : SYN_NOWHERE);
  };
  auto load_x = [&](int s, bf16x8 (&f)[FM]) {
    const unsigned at = x_at + (unsigned)((s / 2) * 256 + (s % 2) * 32) * 2;
#pragma unroll
    for (int j = 0; j < FM; ++j) f[j] = buffer_load16(vx, s < steps ? at + j * w_frag : SYN_NOWHERE);
  };
#pragma unroll
  for (int s = 0; s < S; s += 2) {
    // (in this order: the loop waits for no load that is younger than those it takes, on any way into it)
    load_w(s, wf[s]);
    __builtin_amdgcn_sched_barrier(0);
    load_x(s, xf[s]), load_x(s + 1, xf[s + 1]);
    __builtin_amdgcn_sched_barrier(0);
    load_w(s + 1, wf[s + 1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int s0 = 0; s0 < steps; s0 += S) {
#pragma unroll
    for (int u = 0; u < S; ++u) {
#pragma unroll
      for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(wf[u][i]), "v"(xf[u][j]));
      __builtin_amdgcn_sched_barrier(0);
      load_w(s0 + S + u, wf[u]);
      if (u % 2 == 1) load_x(s0 + S + u - 1, xf[u - 1]), load_x(s0 + S + u, xf[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // (the compiler does not know the matrix instructions for what they are: their results are waited for by hand)
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) asm volatile("" : "+a"(acc[i][j]));
  // fragment f: rows 2 (f / 2 / FM) + f % 2 of W (gate and up side by side), rows f / 2 % FM of x
#pragma unroll
  for (int f = 0; f < FRAGS; ++f) {
    const int q = f / 2;
    part[(wave * FRAGS + f) * SYN_WAVE + lane] = acc[2 * (q / FM) + f % 2][q % FM];
  }
  __syncthreads();
  for (int q = wave; q < FRAGS / 2; q += 4) {
    f32x4 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v[h] = part[(2 * q + h) * SYN_WAVE + lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) v[h] += part[(w * FRAGS + 2 * q + h) * SYN_WAVE + lane];
    }
    const int m = 16 * (q % FM) + r16, n = n0 + 32 * (q / FM) + 4 * g;
    if (m >= M) continue;
    if constexpr (PAIRED) {
      bf16x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = (bf16)gated(ep.act, v[0][e], v[1][e], ep.limit);
      const int col = n0 / 2 + 16 * (q / FM) + 4 * g;
      if (n < N) *(bf16x4*)((bf16*)out + (size_t)m * (N / 2) + col) = r;
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (n + 16 * h >= N) continue;
        const size_t at = ((size_t)blockIdx.y * M + m) * N + n + 16 * h;
        f32x4 o;
        bf16x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = point_activation(ep.point, v[h][e]), r[e] = (bf16)o[e];
        if (ep.out_is_f32) *(f32x4*)((float*)out + at) = o;
        else *(bf16x4*)((bf16*)out + at) = r;
      }
    }
  }
}

template <int NF, int FM, int S, bool PAIRED>
static int launch_rows_tile(const bf16* x, const bf16* wp, void* out, Epilogue ep, int M, int N, int K, int slices, hipStream_t stream) {
  constexpr int LDS = 4 * NF * FM * SYN_WAVE * 16;
  static OncePerDevice raised;
  const hipError_t e = once_per_device(raised, [&] {
    return hipFuncSetAttribute((const void*)gemm_rows_kernel<NF, FM, S, PAIRED>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  SYN_CHECK(e == hipSuccess, "gemm: %d bytes of LDS refused: %s", LDS, hipGetErrorString(e));
  const int k_slice = ((K / 64 + slices - 1) / slices) * 64;
  gemm_rows_kernel<NF, FM, S, PAIRED><<<dim3((N + 16 * NF - 1) / (16 * NF), slices), 256, LDS, stream>>>(x, wp, out, ep, M, N, K, k_slice);
  return 0;
}
// nf: 16-row groups of W a workgroup (2, 4 or 6), picked by the host's rule (ops.rows_tile).  Deeper where few rows of x leave room; six
// groups beside more than 48 rows of x, or four beside more than 96, do not fit the registers with nothing moved between them.
template <bool PAIRED>
static int launch_rows(int nf, const bf16* x, const bf16* wp, void* out, Epilogue ep, int M, int N, int K, int slices, hipStream_t stream) {
  SYN_CHECK(M <= (nf == 6 ? 48 : nf == 4 ? 96 : 128) && (nf == 2 || nf == 4 || nf == 6) && K % 64 == 0 && N % (PAIRED ? 32 : 16) == 0 &&
            (size_t)K * 2 * 128 < 0x7fffffffull, "gemm: %d rows beside %d x 16 of W, N = %d, K = %d", M, nf, N, K);
#define SYN_ROWS(NF, FM, S) return launch_rows_tile<NF, FM, S, PAIRED>(x, wp, out, ep, M, N, K, slices, stream)
  if (nf == 6) {
    if (M <= 16) SYN_ROWS(6, 1, 8);
    if (M <= 32) SYN_ROWS(6, 2, 6);
    SYN_ROWS(6, 3, 4);
  }
  if (nf == 4) {
    if (M <= 16) SYN_ROWS(4, 1, 8);
    if (M <= 32) SYN_ROWS(4, 2, 6);
    if (M <= 48) SYN_ROWS(4, 3, 6);
    if (M <= 64) SYN_ROWS(4, 4, 6);
    SYN_ROWS(4, 6, 4);
  }
  if (M <= 16) SYN_ROWS(2, 1, 8);
  if (M <= 32) SYN_ROWS(2, 2, 6);
  if (M <= 48) SYN_ROWS(2, 3, 6);
  if (M <= 64) SYN_ROWS(2, 4, 6);
  if (M <= 96) SYN_ROWS(2, 6, 4);
  SYN_ROWS(2, 8, 4);
#undef SYN_ROWS
}

// ------------------------------------------------------------------ tiled, M > 64: one stream of k-steps over all tiles
// What bounds it: the matrix units, and under random operands the power that they draw (a product of zeros of
// 2,048 x 24,576 x 4,096 takes 209 us, of random numbers 278).  The kernel therefore spends as little as it can on
// everything else:
//   * four waves, each with a quarter of the tile (128 x 128 of 256 x 256: 256 accumulators, one wave a SIMD): a k-step of
//     64 MFMAs needs 16 fragment reads, two thirds of what eight waves of 128 x 64 need, and no two waves compete for a SIMD;
//   * the accumulators stay where they are: MFMAs are written as statements that read and write the same accumulation
//     registers (given the builtin, the compiler moves some 400 registers around in every turn of the loop);
//   * k-tiles of 32 in a ring of four LDS buffers (up to eight for the smaller tiles, whose k-steps are shorter than the way
//     from memory).  While the MFMAs of a k-step run (operands in registers), the fragments of the next one are read and the
//     loads of the k-tile a ring ahead are issued, evenly between the MFMAs: a burst of loads holds up the wave that
//     issues it (the texture addresser takes about 25 cycles for each);
//   * x comes in whole lines: a load takes 128 bytes of each of 8 rows, two k-tiles at once, into a ring of its own.  Pieces of 64
//     bytes, one k-tile of 16 rows, cost the caches a request each as well and every line twice (2,048 x 24,576 x 4,096, zeros:
//     270 us, in whole lines 231; random numbers 298 -> 291; 1,024 rows 187 -> 169, 512 98 -> 84; 512 x 4,096 x 12,288 65 -> 53;
//     40,960 x 2,560 x 9,728 1,655 -> 1,600; a prompt of 2,048 tokens at the 8B shape 26.75 -> 25.2 ms);
//   * where the loads have got to is kept from step to step: 24 scalar instructions of two steps instead of 39 (of 512 x 6,144 x 4,096
//     in tiles of 64 x 128, whose steps have eight MFMAs, 50.8 -> 40.1 us; 45.2 with x in pieces);
//   * a workgroup goes through several tiles and its loads run ahead into the next one: no tile but the first waits for
//     its first operands, and a tile's stores drain behind the next one's MFMAs;
//   * W's fragment is the first operand, so that a lane's four results are neighbours in a row; two groups of them are joined
//     by a swap between rows of 16 lanes into 16 bytes a lane.  Stores of a large output are marked as streamed past the
//     caches: ordinary ones push x and W out of the L2s (2,048 x 24,576 x 4,096, zeros: 272 us, streamed 216); an output
//     that fits the memory-side cache is stored there for its reader (128 x 4,096 x 12,288 in 8 slices and the norm behind it: 37
//     us streamed, 34 not).
// Against the kernel before it (eight waves of 128 x 64, k-tiles of 64 in two buffers, a tile a workgroup), random operands,
// W in fragment order, with the gated activation: 2,048 x 24,576 x 4,096 335 -> 278 us (1.48 PFLOP/s), 35,901 x 19,456 x
// 2,560 3,056 -> 2,476 us (1.44); without: 8,192 x 24,576 x 4,096 1,313 -> 1,128 us, 35,901 x 2,560 x 9,728 1,533 -> 1,402.
// Operands: W in fragment order (WP: pack_weight) or in plain rows, x in plain rows.  In LDS a row of 32 k-values of W in plain
// rows is four chunks of 16 bytes, slot s of row r holding chunk s ^ (r / 4 % 4), a row of 64 of x eight chunks, slot s holding
// chunk s ^ (r / 2 % 8), so that 16 lanes with the same chunk of 16 rows
// touch every bank once; fragments of W lie as they come.  Rows beyond M or N lie behind the descriptors' ends: they are
// read as zeros without traffic, and their results are dropped by the output's descriptor.

// Tile i in the order in which they are handed out: columns of four tiles of W, along which the rows of x run; 32 in a row
// (8 x 4 tiles) go to the workgroups of one XCD, which then share rows of x and of W in its L2.
struct TileAt {
  int m, n, slice;
};
__device__ __forceinline__ TileAt stream_tile(int i, int tiles_m, int tiles_n) {
  const int per = tiles_m * tiles_n, s = i / per, t = i - s * per;
  const int column = t / (4 * tiles_m), in = t - column * 4 * tiles_m;
  const int w = min(4, tiles_n - 4 * column);
  return {in / w, 4 * column + in % w, s};
}

// OUT: what is stored
#define SYN_OUT_BF16 0
#define SYN_OUT_F32 1
#define SYN_OUT_GATED 2     // W: gate and up rows in turns of 16; bf16, half as wide
// ONCE: the rows fit one tile, so that W is read once: its loads are marked non-temporal.  (A stream of weights through the L2s pushes
// everything else out of them.  Steps with the hint taken from the gated product, ms: 8B shape 64 rows 4.07 -> 4.30, 96 4.70 -> 4.91, 128
// 5.07 -> 5.26, eight layers of the 32B one 64 1.89 -> 2.00, 96 2.00 -> 2.18, 256 2.78 -> 3.10; from q/k/v, o_proj or down_proj of the latter 10 to
// 60 us.  Where several rows of tiles read W it lost: 41,000 tokens at the 4B shape 299 -> 317 ms, 1,733 28.97 -> 29.13, and in two rows of tiles
// 160 tokens at the 8B shape 176 -> 181 us a layer, 96 at the 4B shape 118 -> 125.)
template <int BM, int BN, int OUT, bool WP, bool ONCE>
__global__ void __launch_bounds__(256, 1)
gemm_stream_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, void* __restrict__ out, Epilogue ep,
                   int M, int N, int K, int k_slice, int tiles, int whole, int streamed) {
  constexpr int BK = 32, STAGES = stream_stages(BM, BN), PAIRS = stream_pairs(BM, BN), WAVES = 4;
  constexpr int XL = BM / 32, WL = BN / 64, PASSES = XL / 2 + WL;   // loads of a wave: of a pair of k-tiles of x, of a k-tile of W, a step
  constexpr int FM = BM / 32, FN = BN / 32;                   // fragments of 16 rows that a wave holds of x and of W
  constexpr int NM = FM * FN, NR = FM + FN;                   // MFMAs and fragment reads of a wave in a k-step
  constexpr int READ_EVERY = NM / NR > 3 ? 3 : NM / NR, LOAD_EVERY = NM / PASSES;
  static_assert(BM % 64 == 0 && BN % 64 == 0 && STAGES % 2 == 0 && stream_lds(BM, BN) <= 163840, "tile shape");
  static_assert(READ_EVERY >= 1 && LOAD_EVERY >= 1 && FN % 2 == 0, "reads, loads and stores find their places");
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];   // x [PAIRS][BM][64], W [STAGES][BN][32]
  const int tid = threadIdx.x, lane = tid % SYN_WAVE, grid = (int)gridDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / SYN_WAVE);   // scalar: LDS addresses of the loads stay scalar
  const int wm = (wave / 2) * (BM / 2), wn = (wave % 2) * (BN / 2);
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const size_t row_bytes = (size_t)K * sizeof(bf16);
  int at = ((int)blockIdx.x % 8) * (grid / 8) + (int)blockIdx.x / 8;   // workgroup b runs on XCD b % 8
  if (at >= tiles) return;

  // Load p of x fills tile rows (p * WAVES + wave) * 8 .. + 8, 128 bytes of each; of W rows (p * WAVES + wave) * 16 .. + 16, a fragment as
  // it lies or four rows of 64 bytes at a time
  unsigned src_x[XL], src_w[WL];
#pragma unroll
  for (int p = 0; p < XL; ++p) src_x[p] = (unsigned)((size_t)((p * WAVES + wave) * 8 + lane / 8) * row_bytes + ((lane % 8) ^ (wave % 2 * 4 + lane / 16)) * 16);
#pragma unroll
  for (int p = 0; p < WL; ++p) {
    const int row0 = (p * WAVES + wave) * 16;
    src_w[p] = WP ? (unsigned)((size_t)row0 * row_bytes + lane * 16)
                  : (unsigned)((size_t)(row0 + lane / 4) * row_bytes + ((lane % 4) ^ (lane / 16)) * 16);
  }
  struct Source {      // of a tile: the rows of x and W from its first k-value on, and its k-steps
    BufferView x, w;
    int steps;
  };
  auto source = [&](const TileAt& t) {
    const int m0 = t.m * BM, n0 = t.n * BN, k0 = t.slice * k_slice;
    Source s;
    s.x = buffer_view(x + (size_t)m0 * K + k0, (size_t)(M - m0) * row_bytes - k0 * sizeof(bf16));
    s.w = buffer_view(w + (size_t)n0 * K + (size_t)k0 * (WP ? 16 : 1), (size_t)(N - n0) * row_bytes - (size_t)k0 * sizeof(bf16) * (WP ? 16 : 1));
    s.steps = (min(K, k0 + k_slice) - k0) / BK;
    return s;
  };
  // Where the loads have got to, x's in pairs of k-tiles: the way from here on through this tile and into the next one.  (Kept from step
  // to step, all in bytes: with one wave a SIMD, scalar instructions of a step stand beside its MFMAs, of which the smallest tile has
  // eight.)
  constexpr int W_TILE = BK * (int)sizeof(bf16) * (WP ? 16 : 1), X_PAIR = 2 * BK * (int)sizeof(bf16);
  constexpr int W_BUF = BN * BK * (int)sizeof(bf16), X_BUF = BM * X_PAIR;
  struct Way {
    BufferView v;
    int at, end;
  };
  auto onward = [&](Way& y, int by, const BufferView& then, int then_end) {
    y.at += by;
    if (__builtin_expect(y.at == y.end, 0)) y.v = then, y.at = 0, y.end = then_end;
  };
  const int x_to = wave * 8 * X_PAIR, w_to = PAIRS * X_BUF + wave * 16 * BK * (int)sizeof(bf16);
  auto fetch_x = [&](const Way& y, int xbuf, int p) {
    buffer_to_lds16(y.v, (char*)smem + xbuf + x_to + p * (WAVES * 8 * X_PAIR), src_x[p], y.at);
  };
  auto fetch_w = [&](const Way& y, int buf, int p) {
    buffer_to_lds16<ONCE>(y.v, (char*)smem + buf + w_to + p * (WAVES * 16 * BK * (int)sizeof(bf16)), src_w[p], y.at);
  };
  f32x4 acc[FM][FN];
  const int r16 = lane % 16, q4 = lane / 16;
  // in bytes; the second k-tile of a pair: chunks 4 to 7, bit 2 of the slot
  const int x_at = ((wm + r16) * 2 * BK + (q4 ^ (r16 / 2)) * 8) * 2, x_at2 = x_at ^ 64;
  const int w_at = PAIRS * X_BUF + (WP ? wn * BK + lane * 8 : (wn + r16) * BK + (q4 ^ (r16 / 4)) * 8) * 2;
  bf16x8 a[2][FM], b[2][FN];      // two sets of fragments: one is multiplied while the other is read
  auto read_one = [&](int xbuf, int half, int buf, int set, int idx) {
    if (idx < FM) a[set][idx] = *(const bf16x8*)((const char*)smem + xbuf + (half ? x_at2 : x_at) + idx * 16 * X_PAIR);
    else b[set][idx - FM] = *(const bf16x8*)((const char*)smem + buf + w_at + (idx - FM) * 16 * BK * 2);
  };
  Way way_x, way_w;
  int buf = 0, xbuf = 0, xbuf_before = 0;
  // A k-step over fragment set SET, the step's parity (FRESH: a tile's first): reads the fragments of the next step and asks for W's
  // k-tile a ring ahead and half a pair of x, the second half of the pair begun in the step before or the first one of the pair
  // that takes this pair's buffer, whose fragments are all in registers; near a tile's end they belong to the workgroup's next tile
  auto step = [&](const Source& then, auto set, auto fresh) {
    constexpr int SET = decltype(set)::value;
    const int next = buf + W_BUF == STAGES * W_BUF ? 0 : buf + W_BUF;
    const int xnext = SET ? (xbuf + X_BUF == PAIRS * X_BUF ? 0 : xbuf + X_BUF) : xbuf;
#pragma unroll
    for (int q = 0; q < NM; ++q) {
      const int j = q / FM, i = q % FM;
      if constexpr (decltype(fresh)::value)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[i][j]) : "v"(b[SET][j]), "v"(a[SET][i]));
      else
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(b[SET][j]), "v"(a[SET][i]));
      if (q % LOAD_EVERY == 0 && q / LOAD_EVERY < PASSES) {
        const int p = q / LOAD_EVERY;
        if (p < XL / 2) fetch_x(way_x, SET ? xbuf : xbuf_before, SET ? p : p + XL / 2);
        else fetch_w(way_w, buf, p - XL / 2);
      }
      if (q % READ_EVERY == READ_EVERY - 1 && q / READ_EVERY < NR) read_one(xnext, SET ^ 1, next, SET ^ 1, q / READ_EVERY);
      __builtin_amdgcn_sched_barrier(0);
    }
    onward(way_w, W_TILE, then.w, then.steps * W_TILE);
    if constexpr (SET == 0) onward(way_x, X_PAIR, then.x, then.steps * (X_PAIR / 2));
    else xbuf_before = xbuf, xbuf = xnext;
    buf = next;
  };
  // Before the barrier that ends a step a wave waits until its reads have returned and all but its youngest loads, those of
  // the last STAGES - 2 steps, have landed: behind it the k-tile after the next is whole, and the buffer of this step's tile free.
  // (A tile's stores are younger than the loads that the step behind them waits for, and count like loads.)
  constexpr int YOUNGER = (STAGES - 2) * PASSES;
  auto landed = [&] {
    __builtin_amdgcn_s_waitcnt(0x0070 | (YOUNGER & 15) | ((YOUNGER >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  TileAt t = stream_tile(at, tiles_m, tiles_n);
  bool more = at + grid < tiles;
  TileAt t_next = stream_tile(more ? at + grid : at, tiles_m, tiles_n);   // (behind the last tile: loads that nobody reads)
  Source then = source(t_next);
  {
    const Source now = source(t);
    way_x = {now.x, 0, now.steps * (X_PAIR / 2)}, way_w = {now.w, 0, now.steps * W_TILE};
  }
  // what the steps before the first would have asked for
#pragma unroll
  for (int p = 0; p < XL / 2; ++p) fetch_x(way_x, 0, p);
#pragma unroll
  for (int s = 0; s < STAGES; ++s) {
#pragma unroll
    for (int p = 0; p < XL / 2; ++p) fetch_x(way_x, (s + 1) / 2 * X_BUF, s % 2 ? p : p + XL / 2);
#pragma unroll
    for (int p = 0; p < WL; ++p) fetch_w(way_w, s * W_BUF, p);
    onward(way_w, W_TILE, then.w, then.steps * W_TILE);
    if (s % 2 == 0) onward(way_x, X_PAIR, then.x, then.steps * (X_PAIR / 2));
  }
  xbuf_before = STAGES / 2 * X_BUF;
  int steps = source(t).steps;
  landed();
#pragma unroll
  for (int i = 0; i < NR; ++i) read_one(0, 0, 0, 0, i);
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the first fragments are in registers,
  __builtin_amdgcn_s_barrier();         // everywhere
  __builtin_amdgcn_sched_barrier(0);
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  for (;;) {
    step(then, Even{}, std::true_type{}), landed();
    step(then, Odd{}, std::false_type{}), landed();
    for (int kt = 2; kt < steps; kt += 2) {
      step(then, Even{}, std::false_type{}), landed();
      step(then, Odd{}, std::false_type{}), landed();
    }
    // (the compiler does not know that the statements above are matrix instructions: their results may be read 18 states later)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    // lane: row m = wm + 16 i + r16, columns wn + 16 j + 4 q4 .. + 4 of the tile
    constexpr int ELT = OUT == SYN_OUT_F32 ? 4 : 2, JS = OUT == SYN_OUT_GATED ? 4 : 2;   // fragments that make 32 columns
    const int width = OUT == SYN_OUT_GATED ? N / 2 : N, m0 = t.m * BM + wm;
    const BufferView vo = buffer_view((char*)out + ((size_t)t.slice * M + m0) * width * ELT, m0 < M ? (size_t)(M - m0) * width * ELT : 0);
    auto store_all = [&](auto of) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const unsigned row = (unsigned)(16 * i + r16) * width * ELT;
#pragma unroll
        for (int j = 0; j < FN; ++j) asm volatile("" : "+a"(acc[i][j]));    // (not read any earlier than here)
        if constexpr (OUT == SYN_OUT_F32) {
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int n = t.n * BN + wn + 16 * j + 4 * q4;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = of(acc[i][j][e], 0.f);
            if (whole)
              buffer_store16(vo, __builtin_bit_cast(u32x4, v), n < N ? row + n * 4 : SYN_NOWHERE, streamed);
            else
#pragma unroll
              for (int e = 0; e < 4; ++e) buffer_store4(vo, v[e], n + e < N ? row + (n + e) * 4 : SYN_NOWHERE);
          }
        } else {
#pragma unroll
          for (int j = 0; j < FN; j += JS) {
            constexpr int H = JS / 2;                        // the second group's first fragment, H behind the first's
            const bool two = j + H < FN;
            const int n = (t.n * BN + wn + 16 * j) / H;      // the first group's first column of the output
            const int j2 = two ? j + H : j;
            bf16x4 u, v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              u[e] = (bf16)of(acc[i][j][e], acc[i][j + H - 1][e]);
              v[e] = (bf16)of(acc[i][j2][e], acc[i][j2 + H - 1][e]);
            }
            if (whole) {
              // lanes of the rows of 16 lanes 0 and 2 get 8 neighbours of the first group, those of 1 and 3 of the second
              const u32x2 p = __builtin_bit_cast(u32x2, u), q = __builtin_bit_cast(u32x2, v);
              const auto lo = __builtin_amdgcn_permlane16_swap(p.x, q.x, false, false);
              const auto hi = __builtin_amdgcn_permlane16_swap(p.y, q.y, false, false);
              const int second = q4 & 1, col = n + 16 * second + 8 * (q4 / 2);
              buffer_store16(vo, u32x4{(unsigned)lo[0], (unsigned)hi[0], (unsigned)lo[1], (unsigned)hi[1]},
                             col < width && (two || !second) ? row + col * 2 : SYN_NOWHERE, streamed);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int c = n + 4 * q4 + e;
                buffer_store2(vo, u[e], c < width ? row + c * 2 : SYN_NOWHERE);
                if (two) buffer_store2(vo, v[e], c + 16 < width ? row + (c + 16) * 2 : SYN_NOWHERE);
              }
            }
          }
        }
      }
    };
    // The sums added to what is there (the residual rows; syn_gemm_add): what the tile's rows hold is asked for up to four groups of 16 rows ahead, and
    // always before the stores that would otherwise be waited for with it.  (Four groups beside 256 columns spilled: 8,000 rows of 4,096 x 4,096
    // 283 us with the norm instead of 260.)
    auto add_all = [&] {
      constexpr int AHEAD = FM < 4 ? FM : FN > 6 ? 2 : 4;      // (what the registers hold beside the next tile's first fragments)
      f32x4 have[AHEAD][FN];
      auto place = [&](int i, int j) {
        const int n = t.n * BN + wn + 16 * j + 4 * q4;
        return n < N ? (unsigned)(16 * i + r16) * N * 4 + n * 4 : SYN_NOWHERE;
      };
      auto ask = [&](int i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) have[i % AHEAD][j] = __builtin_bit_cast(f32x4, buffer_load16(vo, place(i, j)));
      };
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) ask(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
        for (int j = 0; j < FN; ++j) buffer_store16(vo, __builtin_bit_cast(u32x4, have[i % AHEAD][j] + acc[i][j]), place(i, j), streamed);
        if (i + AHEAD < FM) ask(i + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if constexpr (OUT == SYN_OUT_GATED) {
      if (ep.act == SYN_ACT_SILU) store_all([&](float g, float u) { return gated_quick<SYN_ACT_SILU, false>(g, u, 0.f); });
      else if (ep.act == SYN_ACT_SWIGLU_LIMIT) store_all([&](float g, float u) { return gated_quick<SYN_ACT_SWIGLU_LIMIT, false>(g, u, ep.limit); });
      else store_all([&](float g, float u) { return gated_quick<SYN_ACT_GELU_TANH, false>(g, u, 0.f); });
    } else {
      if (OUT == SYN_OUT_F32 && ep.add) add_all();
      else if (ep.point == SYN_POINT_NONE) store_all([&](float v, float) { return v; });
      else store_all([&](float v, float) { return point_activation(SYN_POINT_RELU_SQUARED, v); });
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!more) break;
    at += grid, t = t_next, steps = then.steps;
    more = at + grid < tiles;
    t_next = stream_tile(more ? at + grid : at, tiles_m, tiles_n);
    then = source(t_next);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);   // nothing may be on its way into LDS when the workgroup ends
}

// The tiles that the kernel comes in, and the estimate of a product's time that picks one of them and the slices of K.  Three
// things run side by side, and the longest counts most (a norm of order 2): rounds of tiles over the chip at `round` us for 4,096
// of K, 45 % of them whatever stands in the tiles; the matrix units' power, at `power` us for 4,096 of K with a tile on every
// compute unit; and the way of W from memory, which is longer where fewer compute units ask for it.  Rows and columns beyond M
// and N are zeros, which draw next to no power: with 129 rows 19,456 x 2,560 takes 34 us, with 256, the same tiles, 48.  So
// both count by the share of a tile that is filled.  The stores of the output come on top, and where W is read by more than one
// row of tiles, so that it passes through the caches (ONCE above), what it pushes out of them: with 96 and 128 rows gate+up in tiles of 64 x
// 192, by itself the faster one, made a layer take longer than in tiles of 128 x 128: 24,576 x 4,096 by 7.4 and 5.1 us, 23,552 x 4,096 10 and
// 7.5, 22,528 x 5,120 7.3 and 3.5, 24,576 x 6,144 12 and 12; with 160 and 192 rows in tiles of 128 x 192 against 256 x 128 the last of them
// 4 us, the others from 2 less to the same.
// The figures are fitted to 744 sizes, every tile and number of slices, with weights that no cache held: 17 to 3,300 rows, multiples of
// the tiles and others, through N x K = 6144 x 4096, 10240 x 5120, 12288 x 4096, 3072 x 1024, 4096 x 2048, 8192 x 2048, 6144 x 2560 (rounded to
// bf16), 4096 x 4096, 4096 x 12288, 2560 x 4096, 2560 x 9728, 5120 x 8192, 5120 x 25600, 1024 x 4096, 2048 x 8192, 6144 x 2560 (32-bit sums
// in 1 to 8 slices of K and the norm that adds them) and, gated, 24576 x 4096, 19456 x 2560, 51200 x 5120, 8192 x 1024.  What the
// estimate picks takes 0.5 % longer than the fastest on average; 3 % of the sizes lose more than 5 %, 2 of them more than 10 %
// (with x in pieces of 64 bytes and the figures and rules fitted to that, on the same products: 3.8 %, 25 %, 11 %).
struct StreamTile {
  int bm, bn;
  double round, power;
  bool plain;       // also over W in plain rows (the others are compiled for fragment order alone)
};
constexpr int STREAMED_TILES = 10;
struct StreamFit {
  StreamTile tiles[STREAMED_TILES];
  // share of a round that an empty tile takes, us of any product, us a byte: of W, of the output, of W beyond 100 MB that several rows of
  // tiles read, of partial sums beyond the first that their reader adds
  double empty, fixed, weight, store, pushed, reader;
};
static const StreamFit STREAMED = {
    {{256, 256, 86.0, 24.8, true}, {256, 192, 64.6, 26.1, true}, {128, 128, 36.4, 0.0, true}, {192, 256, 69.0, 25.3, false},
     {128, 256, 53.6, 0.0, false}, {256, 128, 49.8, 19.7, false}, {192, 192, 54.7, 22.7, false}, {128, 192, 46.5, 0.0, false},
     {64, 128, 20.5, 13.0, true}, {64, 192, 31.6, 13.7, false}},
    0.453, 0.7, 0.124e-6, 0.208e-6, 0.06e-6, 0.14e-6};
// An earlier fit, of the kernel when it read x in pieces of 64 bytes.  It picks nothing any more, but products that it cut hand on their
// sums in 32 bits, and do so still (syn_gemm_sums_line).
static const StreamFit SUMS_LINE = {
    {{256, 256, 82.9, 33.2, true}, {256, 192, 74.7, 20.6, true}, {128, 128, 38.0, 14.4, true}, {192, 256, 67.0, 24.9, false},
     {128, 256, 56.0, 25.9, false}, {256, 128, 66.6, 22.0, false}, {192, 192, 59.0, 26.9, false}, {128, 192, 45.3, 16.3, false},
     {64, 128, 23.5, 12.2, true}, {64, 192, 38.1, 5.3, false}},
    0.255, 4.5, 0.146e-6, 0.229e-6, 0.0, 0.12e-6};
static int stream_slice(int K, int slices) { return ((K + slices - 1) / slices + 127) / 128 * 128; }
static int stream_last_slice(int K, int slices) { return K - (slices - 1) * stream_slice(K, slices); }
struct StreamPlan {
  int tile;        // -1: none takes this K (k-steps come in pairs, and a slice holds a ring of them at least)
  double us;
};
static StreamPlan plan_stream(const StreamFit& fit, int M, int N, int K, int slices, bool packed, int out_bytes) {
  StreamPlan best = {-1, 1e30};
  if (K % 64) return best;
  const long cus = syn_compute_units();
  const double k = stream_slice(K, slices) / 4096.0;
  for (int i = 0; i < STREAMED_TILES; ++i) {
    const StreamTile& s = fit.tiles[i];
    if ((!packed && !s.plain) || stream_last_slice(K, slices) < 32 * stream_stages(s.bm, s.bn)) continue;
    const long down = (M + s.bm - 1) / s.bm, across = (N + s.bn - 1) / s.bn, tiles = down * across * slices;
    const double filled = (double)M / (double)(down * s.bm) * (double)N / (double)(across * s.bn);
    const double work = (double)((tiles + cus - 1) / cus) * s.round * k * (fit.empty + (1.0 - fit.empty) * filled) + fit.fixed;
    const double power = (double)tiles / cus * s.power * k * filled;
    const double ask = tiles < cus ? cbrt((double)cus / (double)tiles) : 1.0, way = fit.weight * 2.0 * N * K * ask * ask;
    const double pushed = M > s.bm ? fit.pushed * fmax(0.0, 2.0 * N * K - 1e8) : 0.0;
    const double us = sqrt(work * work + way * way + power * power) + fit.store * M * N * slices * out_bytes + pushed;
    if (us < best.us) best = {i, us};
  }
  return best;
}

template <int BM, int BN, int OUT, bool PLAIN>
static int launch_stream(const bf16* x, Weight w, void* out, Epilogue ep, int M, int N, int K, hipStream_t stream, int slices) {
  SYN_CHECK(K % 64 == 0 && stream_last_slice(K, slices) >= 32 * stream_stages(BM, BN) && (PLAIN || w.packed),
            "gemm: %d slices of K = %d do not fit tiles of %d x %d", slices, K, BM, BN);
  const size_t lds = stream_lds(BM, BN);
  static OncePerDevice raised;
  if (lds > 65536) {
    const hipError_t e = once_per_device(raised, [&] {
      hipError_t r = hipSuccess;
      for (const void* k : {(const void*)gemm_stream_kernel<BM, BN, OUT, true, false>, (const void*)gemm_stream_kernel<BM, BN, OUT, true, true>})
        if (r == hipSuccess) r = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if constexpr (PLAIN)
        if (r == hipSuccess)
          r = hipFuncSetAttribute((const void*)gemm_stream_kernel<BM, BN, OUT, false, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      return r;
    });
    SYN_CHECK(e == hipSuccess, "gemm: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
  }
  const long tiles = (long)((M + BM - 1) / BM) * ((N + BN - 1) / BN) * slices;
  SYN_CHECK(tiles < (1L << 30), "gemm: M = %d, N = %d make too many tiles", M, N);
  // every workgroup the same number of tiles, or one fewer: the fewest workgroups that need no further round
  const long cus = syn_compute_units(), rounds = (tiles + cus - 1) / cus;
  // (where a tile has fewer steps than the loads of x run ahead each workgroup has one tile: what its loads reach behind it nobody reads)
  const bool ahead = stream_last_slice(K, slices) >= 32 * (stream_stages(BM, BN) + 2);
  const int grid = (int)(8 * (ahead ? (tiles + 8 * rounds - 1) / (8 * rounds) : (tiles + 7) / 8));
  const int whole = N % 16 == 0 && (uintptr_t)out % 16 == 0;      // stores of 16 bytes
  const size_t bytes = (size_t)slices * M * N * (OUT == SYN_OUT_F32 ? 4 : OUT == SYN_OUT_BF16 ? 2 : 1);
  const int streamed = bytes > (48u << 20);      // (of the 256 MB that the memory-side cache holds, beside x and W)
  const int k_slice = stream_slice(K, slices);
  auto launch = [&](auto kernel) { kernel<<<grid, 256, lds, stream>>>(x, w.p, out, ep, M, N, K, k_slice, (int)tiles, whole, streamed); };
  if (!w.packed) {
    if constexpr (PLAIN) launch(gemm_stream_kernel<BM, BN, OUT, false, false>);
  } else if (M <= BM) {
    launch(gemm_stream_kernel<BM, BN, OUT, true, true>);
  } else {
    launch(gemm_stream_kernel<BM, BN, OUT, true, false>);
  }
  return 0;
}

template <int OUT>
static int launch_stream_as(int tile, const bf16* x, Weight w, void* out, Epilogue ep, int M, int N, int K, hipStream_t stream, int slices) {
  switch (tile) {
    case 0: return launch_stream<256, 256, OUT, true>(x, w, out, ep, M, N, K, stream, slices);
    case 1: return launch_stream<256, 192, OUT, true>(x, w, out, ep, M, N, K, stream, slices);
    case 2: return launch_stream<128, 128, OUT, true>(x, w, out, ep, M, N, K, stream, slices);
    case 3: return launch_stream<192, 256, OUT, false>(x, w, out, ep, M, N, K, stream, slices);
    case 4: return launch_stream<128, 256, OUT, false>(x, w, out, ep, M, N, K, stream, slices);
    case 5: return launch_stream<256, 128, OUT, false>(x, w, out, ep, M, N, K, stream, slices);
    case 6: return launch_stream<192, 192, OUT, false>(x, w, out, ep, M, N, K, stream, slices);
    case 7: return launch_stream<128, 192, OUT, false>(x, w, out, ep, M, N, K, stream, slices);
    case 8: return launch_stream<64, 128, OUT, true>(x, w, out, ep, M, N, K, stream, slices);
    case 9: return launch_stream<64, 192, OUT, false>(x, w, out, ep, M, N, K, stream, slices);
    default: SYN_CHECK(false, "gemm: there is no streamed tile %d", tile);
  }
}

// The tile of gemm_tiled for M > 64: the least rounds over the compute units times the work of a tile; the narrower tiles
// are a fifth less efficient (0 = 256 x 256, 1 = 256 x 192, 2 = 128 x 128, two workgroups a compute unit).
static int pick_register_tile(int M, int N) {
  auto rounds = [](long tiles, long slots) { return (tiles + slots - 1) / slots; };
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const long cus = syn_compute_units();
  const double cost[3] = {(double)rounds(tiles(256, 256), cus) * 256 * 256, (double)rounds(tiles(256, 192), cus) * 256 * 192 * 1.2,
                          (double)rounds(tiles(128, 128), 2 * cus) * 2 * 128 * 128 * 1.2};
  int best = 0;
  for (int i = 1; i < 3; ++i)
    if (cost[i] < cost[best]) best = i;
  return best;
}

// M > 64, gated M > 16, and cut products of 57 rows and more.  A K that the kernel above does not take goes through the tiles that pass through registers (any K that is a multiple
// of 8, one slice) or, in slices, through the smallest of those that load straight into LDS.
template <bool PAIRED>
static int launch_large(const bf16* x, Weight w, void* out, Epilogue ep, int M, int N, int K, hipStream_t stream, int slices = 1, int tile = -1) {
  if (tile < 0) tile = plan_stream(STREAMED, M, N, K, slices, w.packed, PAIRED ? 1 : ep.out_is_f32 ? 4 : 2).tile;
  if (tile >= 0) {
    if (PAIRED) return launch_stream_as<SYN_OUT_GATED>(tile, x, w, out, ep, M, N, K, stream, slices);
    if (ep.out_is_f32) return launch_stream_as<SYN_OUT_F32>(tile, x, w, out, ep, M, N, K, stream, slices);
    return launch_stream_as<SYN_OUT_BF16>(tile, x, w, out, ep, M, N, K, stream, slices);
  }
  if (K % 64 == 0) return launch_direct<128, 128, 64, 2, 4, PAIRED, 3>(x, w, out, ep, M, N, K, stream, slices);
  SYN_CHECK(!w.packed && slices == 1, "gemm: a weight in fragment order, or slices, need a K that is a multiple of 64 (K = %d)", K);
  const int shape = pick_register_tile(M, N);
  if (shape == 0) return launch_tiled<256, 256, 64, 4, 2, PAIRED>(x, w.p, out, ep, M, N, K, stream);
  if (shape == 1) return launch_tiled<256, 192, 64, 4, 2, PAIRED>(x, w.p, out, ep, M, N, K, stream);
  return launch_tiled<128, 128, 64, 2, 2, PAIRED>(x, w.p, out, ep, M, N, K, stream);
}

// Whether an uncut product of 65 to 256 rows goes through the 64 x 128 tiles with k-tiles of 128 (gemm_direct): large weights whose tiles
// go round once (tile_grid, which counts what each XCD gets) and whose last 64 rows are at least half full, where W arrives in longer
// pieces than the streamed tiles ask for.  Direct against the best streamed tile, us: 12,288 x 4,096 with 96 rows 30.4, 32.1, 128 rows
// 32.9, 35.2, 84 rows 34.7, 30.9; 6,144 x 4,096 with 96 rows 27.9, 28.6, 256 rows 30.4, 31.3; 10,240 x 5,120 with 128 rows 40.2, 41.9, 84
// rows 38.1, 36.3; 4,096 x 2,048 with 128 rows 17.1, 13.1; 8,192 x 2,048 17.8, 16.0; 6,144 x 2,560 21.9, 15.9.
// W in plain rows, which the streamed tiles ask for in pieces of 64 bytes of a row, goes through them whatever its size and the rows that
// the last 64 hold: 1,024 x 1,024 9, 11; 2,048 x 2,048 with 96 rows 14, 17, 4,096 x 4,096 27, 38, 128 rows 30, 41, 65 rows 25, 33, 2,560 x 9,728
// with 96 rows 61, 88, 12,288 x 4,096 31, 42; not in two rounds (10,240 x 5,120 with 160 rows 70, 54).
static bool direct_one_round(int M, int N, int K, bool packed) {
  if (M > 256 || K % 128 != 0 || tile_grid(M, N, 64, 128) > syn_compute_units()) return false;
  return !packed || ((M - 1) % 64 >= 31 && K >= 4096 && (long)N * K >= 24L << 20);
}

// The slices of K in which the tiles of 64 or 128 rows by 128 of W that load straight into LDS (gemm_direct) fill the compute units.
static long direct_groups(int M, int N) { return (long)((M + 127) / 128) * ((N + 127) / 128); }
static int direct_slices(int M, int N, int K) {
  const long most = std::min<long>({8, syn_compute_units() / direct_groups(M, N), K / 512});
  int slices = 1;
  while (slices * 2 <= most) slices *= 2;
  return slices;
}

// Whether a cut product of 57 to 64 rows goes through the streamed tiles, in the slices of their estimate: a large W whose tiles of
// gemm_direct leave three eighths of the compute units without work, which slices in other numbers than powers of two reach.  Kernel times
// in a prompt step of 64 rows, us, these tiles and streamed: 5,120 x 25,600 cut in 4 and 6 56.1, 46.5, 10,240 x 5,120 in 2 and 3 26.1, 24.0,
// 5,120 x 8,192 in 4 and 6 21.4, 19.5 (W in fragment order); smaller ones and those that fill them: 6,144 x 4,096 13.6, 14.7, 4,096 x 12,288 21.1, 21.7, 2,560 x
// 9,728 15.9, 17.4, 8,192 x 28,672 in 4 and 8 6 less.  Steps with every product streamed, and so: 8B shape 4.07, 3.95 ms, 4B 3.21, 3.11.
static bool few_rows_streamed(int N, int K, bool packed) {
  return packed && (long)N * K >= 24L << 20 && 8 * direct_groups(64, N) * direct_slices(64, N, K) <= 5L * syn_compute_units();
}

// Whether a cut product goes through the tiles of 128 x 128 that hold k-tiles of 64 (gemm_direct), in slices that are a power of two.  W in
// fragment order: 177 to 256 rows, where their workgroups fill three quarters of the compute units and more and W has 48 to 96 MB (less of
// it the streamed tiles bring in with fewer partial sums, more of it in longer runs).  What a layer of a prompt step gains over the streamed
// tiles, us: 6,144 x 4,096 with 4,096 x 12,288 behind it 0.8 with 192 rows, 4.2 with 256, 6,144 x 6,144 -1.2, -2.0, 8,192 x 6,144 0.5, 2.2,
// 7,168 x 5,120 -0.3, 2.7, 3,072 x 8,192 0.2, -0.9; beyond: 4,096 x 14,336 -3.7, -1.8, 6,144 x 16,384 -20, -20, 8,192 x 28,672 -46, -23; below:
// 4,096 x 4,096 -1.4, -1.0.  (65 to 128 rows gained 1 % of the 8B shape's step on one card and lost 1 to 2 on another.)
// W in plain rows: 65 to 128 rows whatever W (the product and the sum of its slices, these tiles and streamed: 6,144 x 2,560 with 128 rows 20,
// 24, 2,560 x 9,728 with 96 26, 27, 4,608 x 3,584 22, 20), 177 to 256 where they fill the compute units (4,096 x 4,096 with 256 rows 25, 29,
// 8,192 x 4,096 37, 39; 5,120 x 5,120, 160 workgroups, 40, 36).
static bool direct_cut(int M, int N, int K, bool packed) {
  const long w = (long)N * K, groups = direct_groups(M, N), cus = syn_compute_units();
  if (K % 128 != 0 || groups > cus || M <= 64 || M > 256) return false;
  if (M <= 176) return !packed && M <= 128;
  if (packed && (w < 24L << 20 || w > 48L << 20)) return false;
  return 4 * groups * direct_slices(M, N, K) >= 3 * cus;
}

// Into how many slices of K a product of more than 56 rows is cut when its reader adds partial sums: those of the tiles above or, for
// the streamed ones, the smallest estimate of the product's time and of what its reader pays for the slices beyond the first (M x N
// floats each, half of them from caches).
static int plan_slices(const StreamFit& fit, int M, int N, int K, bool packed) {
  int best = 1;
  double least = 1e30;
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  for (int s : {1, 2, 3, 4, 6, 8}) {
    const StreamPlan p = plan_stream(fit, M, N, K, s, packed, 4);
    if (p.tile < 0) break;
    const double us = p.us + (s - 1) * fit.reader * 4.0 * M * N;
    if (us < least) least = us, best = s;
  }
  return best;
}
SYN_EXPORT int syn_gemm_cut_slices(int M, int N, int K, int packed) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  if (M <= 64 ? !few_rows_streamed(N, K, packed) : direct_cut(M, N, K, packed)) return direct_slices(M, N, K);
  return plan_slices(STREAMED, M, N, K, packed);
}

// Whether a product that could be rounded to 16 bits hands on its 32-bit sums whatever number of slices is the fastest now: a line that a
// fit of the tiles' times must not move, since it decides how precise a result is.  (Products that are cut hand them on in any case.  Eight
// layers of the 32B shape with 1,600 tokens, whose q, k and v this concerns: 11.2 ms rounded, 11.4 so, 12.3 when the line was drawn.)
SYN_EXPORT int syn_gemm_sums_line(int M, int N, int K) { return plan_slices(SUMS_LINE, M, N, K, true) > 1; }

// ------------------------------------------------------------------ entry point
// dtype: 0 = float in, float out; 1 = bf16 in, bf16 out; 2 = bf16 in, float out.
// slices > 1 (bf16 in, float out): out is [slices, M, N], slice s holds the sum over its part of K; the
// reader adds the slices.
// w_packed: w is the weight in fragment order (pack_weight; bf16, N a multiple of 16, K of 128): for the tiles that
// load straight into LDS; the other kernels read plain rows only.
// point: what the finished sums pass before they are stored (point_activation; one slice).
// tile: -1, or for tests and measurements one of STREAMED.tiles, whatever the rules below would take (bf16 operands).
// scratch: working memory for 32-bit operands (syn_gemm_f32_scratch floats, or null where that is none).
int launch_gemm_f32(const float* x, const float* w, float* out, int M, int N, int K, int point, float* scratch, int64_t scratch_floats, hipStream_t stream);   // gemm_f32.hip
SYN_EXPORT int syn_gemm(const void* x, const void* w, void* out, int dtype, int M, int N, int K, int force_simt,
                        int slices, int w_packed, int point, int tile, int rows, float* scratch, int64_t scratch_floats, hipStream_t stream) {
  SYN_CHECK(tile < 0 || (dtype != 0 && !force_simt && K % 64 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0),
            "gemm: the streamed tiles take aligned bf16 operands and a K that is a multiple of 64 (K = %d)", K);
  SYN_CHECK(point >= 0 && point < SYN_POINT_COUNT && (point == SYN_POINT_NONE || slices == 1),
            "gemm: activation code %d over %d slices", point, slices);
  SYN_CHECK(M > 0 && N > 0 && K > 0, "gemm: empty shape M=%d N=%d K=%d", M, N, K);
  SYN_CHECK(!w_packed || (dtype != 0 && !force_simt && N % 16 == 0 && K % 128 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0),
            "gemm: a weight in fragment order needs bf16 operands, N = %d a multiple of 16 and K = %d of 128", N, K);
  SYN_CHECK(dtype >= 0 && dtype <= 2, "gemm: unknown dtype code %d", dtype);
  SYN_CHECK(slices >= 1 && (slices == 1 || (dtype == 2 && !force_simt && K % 8 == 0 && slices <= 64 && (M <= 64 || K % 64 == 0))),
            "gemm: %d slices of K need bf16 operands and a float output (and beyond 64 rows a K that is a multiple of 64; K = %d)", slices, K);
  const dim3 simt_grid((N + SIMT_BN - 1) / SIMT_BN, (M + SIMT_BM - 1) / SIMT_BM);
  if (dtype == 0) {
    const float *xf = (const float*)x, *wf = (const float*)w;
    float* of = (float*)out;
    if (!force_simt && K % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0)
      return launch_gemm_f32(xf, wf, of, M, N, K, point, scratch, scratch_floats, stream);
    gemm_simt_kernel<float, float><<<simt_grid, 256, 0, stream>>>(xf, wf, of, M, N, K, point);
    SYN_LAUNCH_CHECK("gemm_simt");
    return 0;
  }
  const int out_is_f32 = dtype == 2;
  const Epilogue ep = {out_is_f32, SYN_ACT_SILU, 0.f, point};   // (no gate in a plain product)
  const bool aligned = (K % 8 == 0) && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0);
  SYN_CHECK(slices == 1 || aligned, "gemm: slices of K need 16-byte aligned operands");
  if (force_simt || !aligned) {
    if (out_is_f32)
      gemm_simt_kernel<bf16, float><<<simt_grid, 256, 0, stream>>>((const bf16*)x, (const bf16*)w, (float*)out, M, N, K,
                                                                  point);
    else
      gemm_simt_kernel<bf16, bf16><<<simt_grid, 256, 0, stream>>>((const bf16*)x, (const bf16*)w, (bf16*)out, M, N, K, point);
    SYN_LAUNCH_CHECK("gemm_simt");
    return 0;
  }
  const bf16* xb = (const bf16*)x;
  const bf16* wb = (const bf16*)w;
  const Weight wt = {wb, w_packed != 0};
  // (from sweeps at the shapes of an 8B model, N = 4096 .. 151936, K = 4096 and 12288, where no other are named)
  int rc = 0;
  if (tile >= 0) {
    rc = launch_large<false>(xb, wt, out, ep, M, N, K, stream, slices, tile);
  } else if (rows && w_packed) {
    rc = launch_rows<false>(rows, xb, wb, out, ep, M, N, K, slices, stream);
  } else if (M == 1 && slices == 1 && !w_packed) {
    // one row: fragments of W straight from memory, K split over the waves
    if (N <= 8192) launch_skinny<1, 16, 4>(xb, wb, out, ep, M, N, K, stream);
    else launch_skinny<1, 8, 4>(xb, wb, out, ep, M, N, K, stream);
  } else if (M <= 32) {
    // few rows: memory-bound; small tiles (many workgroups), deep in K (long pieces of each row), three
    // k-tiles in flight, straight into LDS where K allows it
    if (N >= 65536 && K % 256 == 0) rc = launch_direct<32, 64, 256, 1, 2>(xb, wt, out, ep, M, N, K, stream, slices);
    else if (N >= 65536 && !w_packed) rc = launch_tiled<32, 32, 256, 1, 1>(xb, wb, out, ep, M, N, K, stream, slices);
    else if (K % 128 == 0) rc = launch_direct<32, 64, 128, 1, 2>(xb, wt, out, ep, M, N, K, stream, slices);
    else rc = launch_tiled<32, 64, 128, 1, 2>(xb, wb, out, ep, M, N, K, stream, slices);
  } else if (M <= 64 && K % 128 == 0 && !(M > 56 && slices > 1 && few_rows_streamed(N, K, wt.packed))) {
    // 33 to 64 rows: 128 rows of W a workgroup, so that the rows of x are fetched half as often (every
    // workgroup reads all of x), three k-tiles in a ring, one workgroup a compute unit
    rc = launch_direct<64, 128, 128, 2, 4, false, 3>(xb, wt, out, ep, M, N, K, stream, slices);
  } else if (slices > 1 && direct_cut(M, N, K, wt.packed) && slices == direct_slices(M, N, K)) {
    rc = launch_direct<128, 128, 64, 2, 4, false, 3>(xb, wt, out, ep, M, N, K, stream, slices);
  } else if (M > 64 && slices == 1 && direct_one_round(M, N, K, wt.packed)) {
    rc = launch_direct<64, 128, 128, 2, 4, false, 3>(xb, wt, out, ep, M, N, K, stream);
  } else if (M <= 64 && K % 128 != 0) {
    rc = launch_tiled<64, 64, 128, 2, 2>(xb, wb, out, ep, M, N, K, stream, slices);
  } else {
    rc = launch_large<false>(xb, wt, out, ep, M, N, K, stream, slices);
  }
  if (rc) return rc;
  SYN_LAUNCH_CHECK("gemm");
  return 0;
}

// Rows of the tile of gemm_direct that a gated product of 65 to 256 rows over W in plain rows goes through, 0: the streamed tiles.  One tile
// of rows beside 96 or 128 rows of W each, where these go round once and fill most of the compute units, us, these and streamed: 96 rows,
// 24,576 x 4,096 46, 54, 22,016 x 4,160 45, 53, 20,480 x 5,120 54, 67, 18,944 x 3,584 41, 47, 19,456 x 2,560 35, 37, 16,384 x 2,048 (171 tiles) 28,
// 25, 28,672 x 4,096 (299) 87, 59; 160 rows, 24,576 x 4,096 63, 74, 20,480 x 5,120 74, 102, 28,672 x 4,096 64, 77, 32,768 x 4,096 71, 80, 16,384
// x 2,048 (128 tiles) 39, 26, 51,200 x 5,120 (400) 151, 146.
static int direct_gated_tile(int M, int N, int K) {
  const int cus = syn_compute_units(), by96 = (N + 95) / 96, by128 = (N + 127) / 128;
  if (K % 64 != 0 || K < 2048) return 0;
  if (M <= 128) return 4 * by96 >= 3 * cus && by96 <= cus ? 128 : 0;
  return M <= 256 && 16 * by128 >= 9 * cus && by128 <= cus ? (M <= 192 ? 192 : 256) : 0;
}

// resid[M, N] float += x . w^T (bf16, w in fragment order): a product whose reader adds it to the residual rows adds it itself, so that
// the norm behind it reads 4 bytes a value and writes 2, instead of 8 and 6, and writes no rows of its own.  The same sums, added once, as
// the norm would (float + float).  Product and norm, us, before and so: 41,028 rows, 2,560 x 4,096 1,044 -> 968, 2,560 x 9,728 1,942 ->
// 1,855; 2,048 rows, 4,096 x 4,096 79 -> 73, 8,192 x 4,096 145 -> 137, 2,048 x 2,048 32.0 -> 30.3; 8,000 rows, 4,096 x 12,288 608 -> 592, 1,024 x
// 4,096 74.5 -> 72.8; 512 rows, 5,120 x 512 18.2 -> 17.1.  Not where cutting K gains more: 1,024 rows, 4,096 x 12,288 in 4 slices 105, 121 so.
// syn_gemm_adds: whether there are many rows and the streamed tiles take them (the caller sees to it that K would not be cut: partial sums
// are the norm's to add).
SYN_EXPORT int syn_gemm_adds(int M, int N, int K) {
  return M >= 512 && N > 0 && K > 0 && N % 16 == 0 && K % 128 == 0 && plan_stream(STREAMED, M, N, K, 1, true, 4).tile >= 0;
}
SYN_EXPORT int syn_gemm_add(const void* x, const void* w, float* resid, int M, int N, int K, hipStream_t stream) {
  SYN_CHECK(syn_gemm_adds(M, N, K), "gemm_add: no product of %d x %d rows of %d that adds", M, N, K);
  SYN_CHECK(((uintptr_t)x | (uintptr_t)w | (uintptr_t)resid) % 16 == 0, "gemm_add: operands are not aligned");
  const int rc = launch_large<false>((const bf16*)x, {(const bf16*)w, true}, resid, {1, SYN_ACT_SILU, 0.f, SYN_POINT_NONE, 1}, M, N, K, stream);
  if (rc) return rc;
  SYN_LAUNCH_CHECK("gemm_add");
  return 0;
}

// out[M, N/2] = silu(x . Wg^T) * (x . Wu^T), bf16, where w [N, K] holds the rows of Wg and of Wu in
// turns of 16: rows 32b .. 32b+15 are rows 16b .. 16b+15 of Wg, rows 32b+16 .. 32b+31 those of Wu.
// The activation is applied to the 32-bit sums and rounded once.
// w_packed, tile, rows: as for syn_gemm
SYN_EXPORT int syn_gemm_swiglu(const void* x, const void* w, void* out, int M, int N, int K, int act, float limit,
                               int w_packed, int tile, int rows, hipStream_t stream) {
  SYN_CHECK(tile < 0 || K % 64 == 0, "gemm_swiglu: the streamed tiles take a K that is a multiple of 64 (K = %d)", K);
  SYN_CHECK(M > 0 && N > 0 && K > 0, "gemm_swiglu: empty shape M=%d N=%d K=%d", M, N, K);
  SYN_CHECK(!w_packed || K % 128 == 0, "gemm_swiglu: a weight in fragment order needs K = %d a multiple of 128", K);
  SYN_CHECK(act >= 0 && act < SYN_ACT_COUNT, "gemm_swiglu: unknown activation code %d", act);
  const Epilogue ep = {0, act, limit, SYN_POINT_NONE};
  SYN_CHECK(N % 32 == 0, "gemm_swiglu: %d paired rows are no multiple of 32", N);
  SYN_CHECK(K % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0,
            "gemm_swiglu: K = %d must be a multiple of 8 and the operands 16-byte aligned", K);
  const bf16* xb = (const bf16*)x;
  const bf16* wb = (const bf16*)w;
  int rc = 0;
  const Weight wt = {wb, w_packed != 0};
  if (tile >= 0) {
    rc = launch_large<true>(xb, wt, out, ep, M, N, K, stream, 1, tile);
  } else if (rows && w_packed) {
    rc = launch_rows<true>(rows, xb, wb, out, ep, M, N, K, 1, stream);
  } else if (!w_packed && M > 64 && direct_gated_tile(M, N, K)) {
    const int tile = direct_gated_tile(M, N, K);
    if (tile == 128) rc = launch_direct<128, 96, 64, 4, 1, true, 4>(xb, wt, out, ep, M, N, K, stream);
    else if (tile == 192) rc = launch_direct<192, 128, 64, 2, 2, true, 3>(xb, wt, out, ep, M, N, K, stream);
    else rc = launch_direct<256, 128, 64, 4, 2, true, 3>(xb, wt, out, ep, M, N, K, stream);
  } else if (M > 64 || (M > 16 && K >= 256 && K % 64 == 0 && (w_packed || K % 128 != 0 || (M > 32 && (long)N * K < 12L << 20)))) {
    // the streamed tiles from 17 rows on (W in fragment order, us against the tiles below: 19,456 x 2,560 with 24 rows 26.8 -> 23.3, 64 27.3 ->
    // 26.7, 128 34.9 -> 32.9; 24,576 x 4,096 with 64 45.1 -> 43.6, 96 48.2, 47.9; 51,200 x 5,120 with 32 99 -> 94, 128 166 -> 111; 8,192 x 1,024 with
    // 128 18.6 -> 9.4).  W in plain rows from 65 on, or where K keeps it from the tiles below that load straight into LDS, or where it is small
    // (these tiles and those, 33 to 64 rows: 24,576 x 4,096 50, 38, 12,288 x 4,096 43, 34, 16,384 x 2,048 25, 22, 6,144 x 2,560 30, 25, 8,192 x 1,024
    // 10, 13, 2,048 x 2,048 15, 18; 17 to 32: 24,576 x 4,096 49, 40, 2,560 x 9,728 88, 39, 8,192 x 1,024 10, 9; K = 4,160, 22,016 wide 47, 47,
    // K = 1,088, 8,192 wide 10, 14).
    rc = launch_large<true>(xb, wt, out, ep, M, N, K, stream);
  } else if (M == 1 && !w_packed) {
    // one row: fragments of W straight from memory; eight waves on the gate rows, eight on the up rows
    launch_skinny<2, 8, 4, true>(xb, wb, out, ep, M, N, K, stream);
  } else if (M <= 32) {
    if (N >= 65536 && !w_packed) rc = launch_tiled<32, 32, 256, 1, 1, true>(xb, wb, out, ep, M, N, K, stream);
    else if (K % 128 == 0) rc = launch_direct<32, 64, 128, 1, 2, true>(xb, wt, out, ep, M, N, K, stream);
    else rc = launch_tiled<32, 64, 128, 1, 2, true>(xb, wb, out, ep, M, N, K, stream);
  } else if (K % 128 == 0) {
    rc = launch_direct<64, 128, 128, 2, 2, true, 3>(xb, wt, out, ep, M, N, K, stream);
  } else {
    rc = launch_tiled<64, 64, 128, 2, 2, true>(xb, wb, out, ep, M, N, K, stream);
  }
  if (rc) return rc;
  SYN_LAUNCH_CHECK("gemm_swiglu");
  return 0;
}

// The products above for up to 16 rows of x over wp, a copy of W [N, K] in fragment order (see
// gemm_packed_kernel; N a multiple of 16, K of 32).  out_code: 1 = bf16 [M, N], 2 = float [M, N];
// paired: W holds gate and up rows in turns of 16 and out is bf16 [M, N / 2] = act(gate) * up.
// slices > 1 (float out, not paired): out is [slices, M, N], slice s holds the sum over its part of K.
// The norm between two such products (RowNorm above):
//   ss [M, ss_groups] float (or null): the sums of row m are multiplied by rsqrt(sum(ss[m, :]) / norm_dim + eps);
//   resid [M, N] float (or null; then float sums, one slice, not paired, `out` unused): resid += sums,
//   xs [M, N] bf16 = (gain_offset + gain[n]) * resid, ss_out [M, N / 16] = sums of resid^2 over groups of 16 columns.
// point: as for syn_gemm, or SYN_POINT_SOFTCAP with its cap in `limit`.
// add_rows [M, N], add_vec [N] (or null): added into resid beside the sums.
SYN_EXPORT int syn_gemm_packed_norm(const void* x, const void* wp, void* out, int out_code, int M, int N, int K, int paired,
                                    int act, float limit, int slices, const float* ss, int ss_groups, int norm_dim, float eps,
                                    float* resid, void* xs, float* ss_out, const void* gain, int gain_is_f32,
                                    float gain_offset, const float* add_rows, const float* add_vec, int point,
                                    hipStream_t stream) {
  SYN_CHECK(point >= 0 && point <= SYN_POINT_SOFTCAP && (point == SYN_POINT_NONE || (slices == 1 && !paired && !resid)),
            "gemm_packed: activation code %d belongs to a plain product in one slice", point);
  SYN_CHECK(act >= 0 && act < SYN_ACT_COUNT, "gemm_packed: unknown activation code %d", act);
  SYN_CHECK(point != SYN_POINT_SOFTCAP || limit > 0.f, "gemm_packed: a soft cap of %g", (double)limit);
  SYN_CHECK(slices >= 1 && slices <= 64 && (slices == 1 || (out_code == 2 && !paired)),
            "gemm_packed: %d slices of K need a float output [slices, M, N] and no activation", slices);
  const Epilogue ep = {out_code == 2, act, limit, point};
  SYN_CHECK(M > 0 && M <= 16 && N > 0 && K > 0, "gemm_packed: M = %d (1 .. 16), N = %d, K = %d", M, N, K);
  SYN_CHECK(N % 16 == 0 && K % 32 == 0 && (!paired || N % 32 == 0),
            "gemm_packed: N = %d must be a multiple of 16 (32 for paired rows), K = %d of 32", N, K);
  SYN_CHECK(out_code == 1 || out_code == 2, "gemm_packed: unknown output code %d", out_code);
  SYN_CHECK(!paired || out_code == 1, "gemm_packed: the gated product is stored as bf16");
  SYN_CHECK((uintptr_t)x % 16 == 0 && (uintptr_t)wp % 16 == 0, "gemm_packed: operands must be 16-byte aligned");
  RowNorm rn = {};
  if (ss) {
    SYN_CHECK(ss_groups > 0 && norm_dim > 0, "gemm_packed: %d groups of a row statistic over %d columns", ss_groups, norm_dim);
    rn.ss = ss, rn.ss_groups = ss_groups, rn.inv_dim = 1.f / (float)norm_dim, rn.eps = eps;
  }
  if (resid) {
    SYN_CHECK(!paired && slices == 1 && out_code == 2 && xs && ss_out && gain,
              "gemm_packed: the product before a norm is one slice of float sums with xs, ss_out and a gain");
    rn.resid = resid, rn.xs = (bf16*)xs, rn.ss_out = ss_out, rn.gain = gain, rn.gain_is_f32 = gain_is_f32;
    rn.gain_offset = gain_offset, rn.add_rows = add_rows, rn.add_vec = add_vec;
  }
  const bf16* xb = (const bf16*)x;
  const bf16* wb = (const bf16*)wp;
  // from sweeps at N = 4096 .. 151936, K = 4096 and 12288, 1 and 8 rows
  // gate and up rows of the same outputs: from 5 rows of x on a wave takes both (a fragment of x is then loaded
  // once for two products: a decode step of 8 sequences 3.88 -> 3.80 ms; at one row 3.30 -> 3.31 ms, at four
  // within the differences between boxes).  The same for the narrow products (two groups of rows a wave, twice
  // the slices of K) gained under 1 % at 8 sequences and lost as much at 4.
  if (paired && M >= 5) launch_packed2<16, 2, true>(xb, wb, out, ep, M, N, K, stream, 1, rn);
  else if (paired) launch_packed<2, 8, 4, true>(xb, wb, out, ep, M, N, K, stream, 1, rn);
  else if (N <= 8192) launch_packed<1, 16, 2>(xb, wb, out, ep, M, N, K, stream, slices, rn);
  // very wide (the output head): from 5 rows of x on two groups of rows a wave as well (N = 151936, K = 4096 at 8 rows:
  // 193 -> 182 us; at one row 175 -> 179; three or four groups a wave, or deeper, lose again; N = 10240 in two slices
  // of K: 18.9 -> 20.0 us, so only where W is very wide)
  else if (M >= 5 && N >= 32768) launch_packed2<8, 4>(xb, wb, out, ep, M, N, K, stream, slices, rn);
  else launch_packed<1, 8, 8>(xb, wb, out, ep, M, N, K, stream, slices, rn);
  SYN_LAUNCH_CHECK("gemm_packed");
  return 0;
}

SYN_EXPORT int syn_gemm_packed(const void* x, const void* wp, void* out, int out_code, int M, int N, int K, int paired,
                               int act, float limit, int slices, int point, hipStream_t stream) {
  return syn_gemm_packed_norm(x, wp, out, out_code, M, N, K, paired, act, limit, slices, nullptr, 0, 0, 0.f, nullptr, nullptr,
                              nullptr, nullptr, 0, 0.f, nullptr, nullptr, point, stream);
}
