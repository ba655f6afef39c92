// out[M, N] = x[M, K] . W[N, K]^T of 32-bit operands, on the matrix units' 16-bit instructions.
//
// v_mfma_f32_16x16x4_f32 makes 256 multiply-adds a clock and compute unit (149 TFLOP/s of a large product here), the bf16 instructions
// sixteen times as many.  A 32-bit number is the sum of three bf16 numbers (24 bits of mantissa in three times 8, each part the rounded
// rest), the product of two is the sum of nine products of parts, which the matrix units multiply exactly and add in 32 bits,
// and the three of them below 2^-24 of the product are left out: six bf16 products in the place of one, a sixth of the bf16 rate, which is
// more than the 32-bit rate.  The five smaller ones have sums of their own, so that they are not rounded at the size of the first, and
// a chain of 32 k-values rounds once where the 32-bit instruction rounds eight times.  Errors against 64 bits (2-norm over 2-norm, normal
// operands; this, the 32-bit instruction in the same classes): K = 64 4.7e-8, 10.5e-8; 512 8.6e-8, 12.8e-8; 2,560 1.0e-7, 2.4e-7; 9,728
// 1.6e-7, 4.5e-7; positive operands 0.6e-7, 0.75e-7 and 0.6e-7, 1.0e-7 at the last two; products of the size of 1e-35 like those of one.
// An operand that is no number, infinite, or rounds to a bf16 infinity makes some part of a sum none, and the matrix units take parts below
// 2^-126 for zero, so that numbers below 2^-109 lose some of their own: a result that is no finite number, or is not zero and below 2^-90, is
// summed again, term by term (plain_dot), and is what fused multiply-adds in 32 bits give.
//
// The order of the sums is the same whatever the number of rows and the kernel, so a row's results do not depend on what else is in
// the batch: K in chunks of 32, chunk c of class c % 16; the chunks of a class one after another in ascending order into two sums (the
// first products, the five others from the smallest on), which are added; then four classes one after another make a group, and
// the groups one after another the result.
//
//   gemm_f32_few    few rows of x where tiles would leave the chip idle: W streamed once for every 16 of them, a class a wave
//   gemm_f32_tiles  else: tiles through LDS over the parts of x that split_rows has made; where they are few, a workgroup takes one
//                   group of K and add_groups adds the groups' sums
#include <algorithm>
#include <type_traits>
#include "common.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Eight numbers in three parts each: v = p[0] + p[1] + p[2].
__device__ __forceinline__ void split3(const f32x4& lo, const f32x4& hi, bf16x8 (&p)[3]) {
  u32x4 u[3];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f32x2 v = e < 2 ? f32x2{lo[2 * e % 4], lo[2 * e % 4 + 1]} : f32x2{hi[2 * e % 4], hi[2 * e % 4 + 1]};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const unsigned b = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
      u[i][e] = b;
      v = f32x2{v.x - __builtin_bit_cast(float, b << 16), v.y - __builtin_bit_cast(float, b & 0xffff0000u)};
    }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) p[i] = __builtin_bit_cast(bf16x8, u[i]);
}

// Whether the parts' sum v does not stand for the result, and the result then.
__device__ __forceinline__ bool sum_again(float v) { return !(fabsf(v) < INFINITY) || (fabsf(v) < 0x1p-90f && v != 0.f); }
__device__ __attribute__((noinline)) float plain_dot(const float* x, const float* w, int K) {
  float s = 0.f;
  for (int k = 0; k < K; ++k) s = fmaf(x[k], w[k], s);
  return s;
}

#define F32_CLASSES 16
#define F32_GROUPS 4
#define F32_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0)

// Bound by reading W, which no cache holds.  A workgroup owns 16 rows of W and of x; its 16 waves take a class each, U loads of 16 k-values at a
// time, so that the workgroup has up to 128 KB of W under way; both operands are split in registers (88 vector instructions for 2 KB
// of W, two fifths of what a compute unit issues meanwhile), and the classes' sums are added in LDS.
// D[n = 4 (lane / 16) + j][m = lane % 16].  2,560 x 9,728: 1 row 38.5 -> 36.9 us, 16 rows 50.3 -> 49.1 (with the 32-bit instruction, so).
template <int U>
__global__ void __launch_bounds__(16 * SYN_WAVE)
gemm_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N, int K, int point) {
  constexpr int WAVES = F32_CLASSES;
  static_assert(U % 2 == 0, "chunks of 32");
  __shared__ f32x4 part[WAVES][SYN_WAVE];
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE, r16 = lane % 16, k4 = 4 * (lane / 16);
  const int n0 = (int)blockIdx.x * 16;
  // (rows of W beyond N and of x beyond M repeat the last one: their results are never stored)
  const float* wr = w + (size_t)min(n0 + r16, N - 1) * K + k4;
  const int m0 = (int)blockIdx.y * 16;
  const float* xr = x + (size_t)min(m0 + r16, M - 1) * K + k4;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc = zero, low = zero;
  for (int k0 = wave * 32; k0 < K; k0 += WAVES * 16 * U) {
    f32x4 b[U], a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u / 2 * WAVES * 32 + u % 2 * 16;
      const bool in = k + k4 < K;      // (K is a multiple of 4)
      b[u] = in ? __builtin_nontemporal_load((const f32x4*)(wr + k)) : zero;
      a[u] = in ? *(const f32x4*)(xr + k) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; u += 2) {
      if (k0 + u / 2 * WAVES * 32 >= K) break;
      bf16x8 wp[3], xp[3];
      split3(b[u], b[u + 1], wp);
      split3(a[u], a[u + 1], xp);
      low = F32_MFMA(wp[0], xp[2], low);
      low = F32_MFMA(wp[1], xp[1], low);
      low = F32_MFMA(wp[0], xp[1], low);
      low = F32_MFMA(wp[2], xp[0], low);
      low = F32_MFMA(wp[1], xp[0], low);
      acc = F32_MFMA(wp[0], xp[0], acc);
    }
  }
  part[wave][lane] = acc + low;
  __syncthreads();
  if (wave >= 4) return;      // (four waves, one value of a lane's four each)
  float v = 0.f;
#pragma unroll
  for (int g = 0; g < F32_GROUPS; ++g) {
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < WAVES / F32_GROUPS; ++c) s += part[g * (WAVES / F32_GROUPS) + c][lane][wave];
    v += s;
  }
  const int m = m0 + r16, n = n0 + k4 + wave;
  if (m < M && n < N) {
    if (__builtin_expect(sum_again(v), 0)) v = plain_dot(x + (size_t)m * K, w + (size_t)n * K, K);
    out[(size_t)m * N + n] = point_activation(point, v);
  }
}

// x in parts, in the order of the fragments that the tiles multiply: [M / 16][K / 32][part][64 lanes][8], lane r16 + 16 q with k-values
// 4 q .. + 4 and 16 + 4 q .. + 4 of row r16; zeros beyond M and K.
__global__ void __launch_bounds__(256)
split_rows_kernel(const float* __restrict__ x, bf16* __restrict__ xs, int M, int K, int nk) {
  const int lane = threadIdx.x % SYN_WAVE, kt = (int)blockIdx.x * 4 + threadIdx.x / SYN_WAVE, row = (int)blockIdx.y * 16 + lane % 16;
  if (kt >= nk) return;
  const int k = kt * 32 + 4 * (lane / 16);
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
  if (row < M && k < K) lo = *(const f32x4*)(x + (size_t)row * K + k);
  if (row < M && k + 16 < K) hi = *(const f32x4*)(x + (size_t)row * K + k + 16);
  bf16x8 p[3];
  split3(lo, hi, p);
#pragma unroll
  for (int i = 0; i < 3; ++i) *(bf16x8*)(xs + (((size_t)blockIdx.y * nk + kt) * 3 + i) * 512 + lane * 8) = p[i];
}

// Which tile of a product that the matrix units bound: every XCD gets as many as every other (to one tile), a run of the tiles in
// bands of at most eight rows of tiles, all bands alike, column after column of a band.  In panels of 8 x 4 (tile_of_workgroup) the
// XCDs' shares differ by a panel, and all panels of a short last band can go to the same ones: 640 rows of 19,456 x 2,560 837 ->
// 524 us, 384 rows of 2,560 x 9,728 263 -> 180, 192 rows 180 -> 147.
__device__ __forceinline__ bool tile_of_share(int M, int N, int BM, int BN, int& tm, int& tn) {
  const int tiles_n = (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM, tiles = tiles_m * tiles_n;
  const int bands = (tiles_m + 7) / 8, high = (tiles_m + bands - 1) / bands;
  const int xcd = (int)blockIdx.x % 8, local = (int)blockIdx.x / 8, more = tiles % 8;
  if (local >= tiles / 8 + (xcd < more)) return false;
  const int t = xcd * (tiles / 8) + min(xcd, more) + local, band = t / (high * tiles_n), in_band = t - band * high * tiles_n;
  const int rows = min(high, tiles_m - band * high);
  tm = band * high + in_band % rows;
  tn = in_band / rows;
  return true;
}
static int share_grid(int M, int N, int BM, int BN) { return (((M + BM - 1) / BM) * ((N + BN - 1) / BN) + 7) / 8 * 8; }

// Tiles of BM x BN, WN waves side by side with all BM rows each (W is split once, in registers, 7 / FM vector instructions a matrix
// instruction), k-tiles of 32 in a ring of STAGES LDS buffers that loads fill without passing through registers.  A wave's matrix
// instructions take a k-tile's parts of x from the last to the first, and the parts of the next k-tile are read into the registers
// that have become free, so that no wave waits for LDS.
// What bounds many rows: the matrix units' power (six 16-bit products: 242 TFLOP/s of 32 bits at 1.45 PFLOP/s) with the splitting of W
// beside it, and 28 KB a k-tile from the L2s (of a 64 x 128 tile; parts of x take 6 bytes a value): 490 rows of 19,456 x 2,560 take 209 us
// without loads and splits, 247 with these and a sixth of the products, 295 in all (435 with the 32-bit instruction); 1,000 rows 821 ->
// 570.  Few rows: the chain of a k-tile (0.4 to 0.9 us), so K is cut where tiles are few: 64 rows of 2,560 x 9,728 133 -> 54 us.
// D[n = 4 (lane / 16) + e][m = lane % 16].
template <int BM, int BN, int WN, int STAGES, int OCC>
__global__ void __launch_bounds__(64 * WN, OCC)
gemm_f32_tiles_kernel(const bf16* __restrict__ xs, const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out,
                      float* __restrict__ parts, int M, int N, int K, int point) {
  constexpr int BK = 32, WAVES = WN, XL = BM / 16 * 3, WL = BN / 8, PASSES = (XL + WL + WAVES - 1) / WAVES, STAGE = PASSES * WAVES * 1024;
  constexpr int FM = BM / 16, FN = BN / WN / 16, OF_GROUP = F32_CLASSES / F32_GROUPS;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x % SYN_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SYN_WAVE), r16 = lane % 16, q = lane / 16;
  const int wn = wave * (BN / WN);
  int tm, tn;
  if (!tile_of_share(M, N, BM, BN, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN, nk = (K + BK - 1) / BK;
  const size_t row_bytes = (size_t)K * sizeof(float), group_bytes = (size_t)nk * 3072;
  const BufferView vx = buffer_view((const char*)xs + (size_t)(m0 / 16) * group_bytes, (size_t)((M + 15) / 16 - m0 / 16) * group_bytes);
  const BufferView vw = buffer_view(w + (size_t)n0 * K, (size_t)(N - n0) * row_bytes);
  // load l of a k-tile: a fragment of a part of x, or 8 rows of W, whose 16-byte chunks are swizzled
  auto chunk = [&](int row) { return ((lane % 8) ^ (row >> 1)) & 7; };
  unsigned src[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int l = p * WAVES + wave, row = (l - XL) * 8 + lane / 8;
    src[p] = l < XL        ? (unsigned)((l / 3) * group_bytes + (l % 3) * 1024 + lane * 16)
             : l < XL + WL ? (unsigned)((size_t)row * row_bytes + chunk(row) * 16)
                           : SYN_NOWHERE;
  }
  auto fetch = [&](int kt, int buf) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int l = p * WAVES + wave;
      char* to = smem + buf * STAGE + l * 1024;
      if (l < XL) {
        buffer_to_lds16(vx, to, src[p], kt * 3072);
      } else {
        // (where K is no multiple of 32 the last k-tile's chunks behind K are zeros)
        const unsigned s = K - kt * BK < BK && 4 * chunk((l - XL) * 8 + lane / 8) >= K - kt * BK ? SYN_NOWHERE : src[p];
        buffer_to_lds16(vw, to, s, kt * BK * 4);
      }
    }
  };
  // the k-tiles of this workgroup, class by class: those of all groups, or of one
  const int first = parts ? (int)blockIdx.y * OF_GROUP : 0, last = parts ? first + OF_GROUP : F32_CLASSES;
  int steps = 0;
  for (int c = first; c < last; ++c) steps += c < nk ? (nk - c + F32_CLASSES - 1) / F32_CLASSES : 0;
  struct Place {
    int kt, of_class;
  };
  auto next = [&](Place p) { return p.kt + F32_CLASSES < nk ? Place{p.kt + F32_CLASSES, p.of_class} : Place{p.of_class + 1, p.of_class + 1}; };
  f32x4 acc[FM][FN] = {}, low[FM][FN] = {}, sum[FM][FN] = {}, total[FM][FN] = {};
  Place load = {first, first}, at = {first, first};
#pragma unroll
  for (int t = 0; t < STAGES; ++t)
    if (t < steps) fetch(load.kt, t), load = next(load);
  const int x_at = lane * 16;
  int w_at[2];      // k-values 4 q .. + 4 and 16 + 4 q .. + 4 of row r16
  w_at[0] = XL * 1024 + (wn + r16) * 128 + ((q ^ ((wn + r16) >> 1)) & 7) * 16, w_at[1] = w_at[0] ^ 64;
  bf16x8 xp[FM][3], wp[FN][3];
  f32x4 raw[FN][2];
  auto read_x = [&](const char* b, int p) {
#pragma unroll
    for (int j = 0; j < FM; ++j) xp[j][p] = *(const bf16x8*)(b + x_at + (j * 3 + p) * 1024);
  };
  auto read_w = [&](const char* b) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) raw[j][h] = *(const f32x4*)(b + w_at[h] + j * 2048);
  };
  auto split_w = [&] {
#pragma unroll
    for (int j = 0; j < FN; ++j) split3(raw[j][0], raw[j][1], wp[j]);
  };
  auto product = [&](f32x4 (&to)[FM][FN], int wi, int xi) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i) to[i][j] = F32_MFMA(wp[j][wi], xp[i][xi], to[i][j]);
  };
  // this wave's reads have returned and all but its `younger` youngest k-tiles have landed; behind the barrier everyone's
  auto landed = [&](auto younger, bool all) {
    constexpr int Y = decltype(younger)::value * PASSES;
    static_assert(Y < 64, "the counter of loads");
    if (all) __builtin_amdgcn_s_waitcnt(0x0070);
    else __builtin_amdgcn_s_waitcnt(0x0070 | (Y & 15) | (Y >> 4 << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  landed(std::integral_constant<int, STAGES - 1>{}, steps < STAGES);
  read_x(smem, 2), read_x(smem, 1), read_x(smem, 0), read_w(smem);
  split_w();
  int buf = 0;
  for (int i = 0; i < steps; ++i) {
    // the next k-tile is whole and this one's fragments are in registers everywhere: its buffer is free
    landed(std::integral_constant<int, STAGES - 2>{}, i + STAGES > steps);
    if (i + STAGES < steps) fetch(load.kt, buf), load = next(load);
    buf = buf + 1 == STAGES ? 0 : buf + 1;
    const char* b = smem + buf * STAGE;      // (behind the last k-tile: an older one, which nothing multiplies)
    read_w(b);
    product(low, 0, 2);
    __builtin_amdgcn_sched_barrier(0);
    read_x(b, 2);
    product(low, 1, 1), product(low, 0, 1);
    __builtin_amdgcn_sched_barrier(0);
    read_x(b, 1);
    product(low, 2, 0), product(low, 1, 0), product(acc, 0, 0);
    split_w();
    __builtin_amdgcn_sched_barrier(0);
    read_x(b, 0);
    const Place behind = next(at);
    if (behind.of_class != at.of_class) {
#pragma unroll
      for (int ia = 0; ia < FM; ++ia)
#pragma unroll
        for (int j = 0; j < FN; ++j) sum[ia][j] += acc[ia][j] + low[ia][j], acc[ia][j] = low[ia][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (behind.of_class % OF_GROUP == 0 || behind.of_class >= nk) {
#pragma unroll
        for (int ia = 0; ia < FM; ++ia)
#pragma unroll
          for (int j = 0; j < FN; ++j) total[ia][j] += sum[ia][j], sum[ia][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    at = behind;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
  float* to = parts ? parts + (size_t)blockIdx.y * M * N : out;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + 16 * i + r16, n = n0 + wn + 16 * j + 4 * q + e;
        if (m < M && n < N) {
          float v = total[i][j][e];
          if (!parts) {
            if (__builtin_expect(sum_again(v), 0)) v = plain_dot(x + (size_t)m * K, w + (size_t)n * K, K);
            v = point_activation(point, v);
          }
          to[(size_t)m * N + n] = v;
        }
      }
}

// The groups' sums one after another.
__global__ void __launch_bounds__(256)
add_groups_kernel(const float* __restrict__ parts, const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N,
                  int K, int point) {
  const size_t at = (size_t)blockIdx.x * 256 + threadIdx.x, all = (size_t)M * N;
  if (at >= all) return;
  float v = 0.f;
#pragma unroll
  for (int g = 0; g < F32_GROUPS; ++g) v += parts[g * all + at];
  if (__builtin_expect(sum_again(v), 0)) v = plain_dot(x + at / N * K, w + at % N * K, K);
  out[at] = point_activation(point, v);
}

// ------------------------------------------------------------------ which kernel
// A product of M rows in tiles of bm x bn, a step of K by 32 taking `step` us for each tile that a compute unit has and `alone` for the first.
struct F32Tile {
  int bm, bn;
  double alone, step;
};
static const F32Tile F32_TILES[] = {{64, 128, 0.91, 0.80}, {64, 64, 0.59, 0.46}, {32, 128, 0.68, 0.50}, {32, 64, 0.46, 0.272}, {16, 64, 0.40, 0.198}};
constexpr int F32_FEW = -1, F32_ROWS = 2048;      // (the parts of x are kept for so many rows at a time)
struct F32Plan {
  int tile;
  bool cut;
};

// The smallest estimate.  Tiles: steps of a compute unit's tiles side by side, the way of W from memory at 5.7 TB/s, whichever is longer
// counting most, 3 us for the parts of x, and where K is cut 5 us and the way of the groups' sums through memory.  Few rows: W's way at 2.95
// TB/s, 2 % longer a row, for every 16 rows; up to 1 MB of W takes about 3 us whatever the kernel.  Fitted to 58 products of 1 to 1,000 rows, 6,144 x 2,560, 2,560 x 4,096, 19,456 x 2,560, 2,560 x 9,728 and 151,936 x
// 2,560, every tile, cut and whole: what it picks takes 2 % longer than the fastest on average, 14 % at most.  Against the 32-bit
// instruction (its tiles and rules; this), us: 2,560 x 4,096 with 1 row 17, 16, 17 rows 26, 24, 64 55, 29, 300 80, 59, 490 116, 93; 6,144 x 2,560
// 24, 21, 34, 24, 43, 32, 100, 83, 142, 113; 2,560 x 9,728 39, 37, 63, 43, 133, 54, 181, 111, 265, 187; 19,456 x 2,560 56, 42, 58, 49, 78, 74, 268,
// 201, 435, 308; 151,936 x 2,560 with 1 row 286, 275, 17 290, 290, 32 310, 300, 64 493, 376.
static F32Plan plan_f32(int M, int N, int K) {
  F32Plan best = {F32_FEW, false};
  if (M <= 64 && (int64_t)N * K <= 1 << 18) return best;      // (asked before anything that costs the host time: a layer of few tokens plans a dozen times)
  const double cus = syn_compute_units(), w = 4e-6 * N * K;
  double least = M <= 64 ? 3.0 + w / 2.95 * ((M + 15) / 16) * (1.0 + 0.02 * std::min(M, 16)) : 1e30;
  const int nk = (K + 31) / 32;
  for (int i = 0; i < (int)(sizeof(F32_TILES) / sizeof(F32_TILES[0])); ++i)
    for (int cut = 0; cut < 2; ++cut) {
      const F32Tile& t = F32_TILES[i];
      const double tiles = (double)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * (cut ? F32_GROUPS : 1);
      const double even = std::max(1.0, tiles / cus), load = even + 0.25 * (ceil(even) - even);
      const double steps = (cut ? (nk + F32_GROUPS - 1) / F32_GROUPS : nk) * (t.step * (load - 1.0) + t.alone), way = w / 5.7;
      const double us = sqrt(sqrt(steps * steps * steps * steps + way * way * way * way)) + 3.0 + (cut ? 5.0 + 6.4e-6 * M * N : 0.0);
      if (us < least) least = us, best = {i, cut != 0};
    }
  return best;
}

static int64_t f32_parts_of_x(int M, int K) { return (int64_t)((M + 15) / 16) * ((K + 31) / 32) * 768; }     // in floats
static int64_t f32_scratch(int M, int N, int K) {
  const F32Plan p = plan_f32(M, N, K);
  return p.tile == F32_FEW ? 0 : f32_parts_of_x(M, K) + (p.cut ? (int64_t)F32_GROUPS * M * N : 0);
}
// Floats of working memory that syn_gemm needs for 32-bit operands of these sizes, 16-byte aligned (0: none).
SYN_EXPORT int64_t syn_gemm_f32_scratch(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 4) return 0;
  const int rest = M % F32_ROWS;
  return std::max(M >= F32_ROWS ? f32_scratch(F32_ROWS, N, K) : 0, rest ? f32_scratch(rest, N, K) : 0);
}

template <int BM, int BN, int WN, int STAGES, int OCC>
static int launch_f32_tiles(const bf16* xs, const float* x, const float* w, float* out, float* parts, int M, int N, int K, int point, hipStream_t stream) {
  constexpr int LDS = STAGES * ((BM / 16 * 3 + BN / 8 + WN - 1) / WN * WN) * 1024;
  static OncePerDevice raised;
  const auto kernel = gemm_f32_tiles_kernel<BM, BN, WN, STAGES, OCC>;
  if (LDS > 65536) {
    const hipError_t e = once_per_device(raised, [&] { return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS); });
    SYN_CHECK(e == hipSuccess, "gemm: %d bytes of LDS refused: %s", LDS, hipGetErrorString(e));
  }
  kernel<<<dim3(share_grid(M, N, BM, BN), parts ? F32_GROUPS : 1), 64 * WN, LDS, stream>>>(xs, x, w, out, parts, M, N, K, point);
  return 0;
}

// 32-bit operands, 16-byte aligned, K a multiple of 4; scratch: syn_gemm_f32_scratch.
int launch_gemm_f32(const float* x, const float* w, float* out, int M, int N, int K, int point, float* scratch, int64_t scratch_floats, hipStream_t stream) {
  for (int m0 = 0; m0 < M; m0 += F32_ROWS) {
    const int rows = std::min(M - m0, F32_ROWS), nk = (K + 31) / 32, groups = (rows + 15) / 16;
    const float* xm = x + (size_t)m0 * K;
    float* to = out + (size_t)m0 * N;
    const F32Plan plan = plan_f32(rows, N, K);
    if (plan.tile == F32_FEW) {
      gemm_f32_few_kernel<8><<<dim3((N + 15) / 16, groups), F32_CLASSES * SYN_WAVE, 0, stream>>>(xm, w, to, rows, N, K, point);
      continue;
    }
    SYN_CHECK(scratch && (uintptr_t)scratch % 16 == 0 && scratch_floats >= f32_scratch(rows, N, K),
              "gemm: %lld floats of working memory for %d x %d x %d, %lld needed", (long long)scratch_floats, rows, N, K, (long long)f32_scratch(rows, N, K));
    bf16* xs = (bf16*)scratch;
    float* parts = plan.cut ? scratch + f32_parts_of_x(rows, K) : nullptr;
    split_rows_kernel<<<dim3((nk + 3) / 4, groups), 256, 0, stream>>>(xm, xs, rows, K, nk);
    int rc = 0;
    switch (plan.tile) {
      case 0: rc = launch_f32_tiles<64, 128, 4, 2, 2>(xs, xm, w, to, parts, rows, N, K, point, stream); break;
      case 1: rc = launch_f32_tiles<64, 64, 4, 3, 2>(xs, xm, w, to, parts, rows, N, K, point, stream); break;
      case 2: rc = launch_f32_tiles<32, 128, 4, 3, 2>(xs, xm, w, to, parts, rows, N, K, point, stream); break;
      case 3: rc = launch_f32_tiles<32, 64, 4, 3, 3>(xs, xm, w, to, parts, rows, N, K, point, stream); break;
      default: rc = launch_f32_tiles<16, 64, 4, 4, 3>(xs, xm, w, to, parts, rows, N, K, point, stream); break;
    }
    if (rc) return rc;
    if (parts) add_groups_kernel<<<(unsigned)(((size_t)rows * N + 255) / 256), 256, 0, stream>>>(parts, xm, w, to, rows, N, K, point);
  }
  SYN_LAUNCH_CHECK("gemm_f32");
  return 0;
}
