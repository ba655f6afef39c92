// Sampling on the device: one block a row of logits [rows, V] (32-bit).
//   temperature <= 0: argmax, the last of equal maxima
//                     (crates/synaptix-infer/src/sampling/greedy.rs:7-13: Rust's max_by keeps the last)
//   temperature  > 0: x = logit / T (skipped for T == 1), p = softmax(x), the first i with u < cumsum_i,
//                     else the last index that is not -inf (crates/synaptix-infer/src/sampling/multinomial.rs:7-28,
//                     logit_processor.rs:8-18; a dropped entry is never drawn, where the reference falls back to the last index)
// The uniform number u comes from the host (a Philox stream per sequence).
// The reference samples on the host from a downloaded vector; the arithmetic is the same,
// only the order of the two sums differs (parallel instead of sequential).
#include <type_traits>

#include "common.h"

#define SAMPLE_THREADS 1024
#define DRAW_PART 32
#define DRAW_DIRECT 16      // entries of a chunk up to which it is not passed through LDS

struct ArgBest {
  float v;
  int i;
};

__device__ __forceinline__ ArgBest arg_better(ArgBest a, ArgBest b) {
  // larger value wins; of equal values the larger index wins
  if (b.v > a.v || (b.v == a.v && b.i > a.i)) return b;
  return a;
}

__device__ __forceinline__ ArgBest block_argmax(ArgBest best, ArgBest* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    ArgBest o;
    o.v = __shfl_xor(best.v, off, SYN_WAVE);
    o.i = __shfl_xor(best.i, off, SYN_WAVE);
    best = arg_better(best, o);
  }
  constexpr int nw = SAMPLE_THREADS / SYN_WAVE;     // (known, so that the reads below are under way together)
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = best;
  __syncthreads();
  ArgBest r = red[0];
#pragma unroll
  for (int w = 1; w < nw; ++w) r = arg_better(r, red[w]);
  return r;
}

__global__ void __launch_bounds__(SAMPLE_THREADS)
sample_rows_kernel(const float* __restrict__ logits, const float* __restrict__ temperature,
                   const float* __restrict__ uniform, int* __restrict__ out, int V) {
  __shared__ ArgBest red_arg[16];
  __shared__ float red[16];
  __shared__ float chunk_sum[SAMPLE_THREADS];
  __shared__ int found[16];
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* x = logits + (size_t)row * V;
  const float T = temperature ? temperature[row] : 0.f;

  ArgBest best = {-INFINITY, -1};
  if (V % 4 == 0 && (uintptr_t)logits % 16 == 0) {
    // 16-byte loads, four of them in flight: the row is read once, at memory speed
    const float4* x4 = (const float4*)x;
    const int V4 = V / 4, step = blockDim.x;
    for (int i0 = tid; i0 < V4; i0 += 4 * step) {
      float4 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[q] = i0 + q * step < V4 ? x4[i0 + q * step] : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = 4 * (i0 + q * step);
        if (i0 + q * step < V4) {
          best = arg_better(best, ArgBest{v[q].x, i});
          best = arg_better(best, ArgBest{v[q].y, i + 1});
          best = arg_better(best, ArgBest{v[q].z, i + 2});
          best = arg_better(best, ArgBest{v[q].w, i + 3});
        }
      }
    }
  } else {
    for (int i = tid; i < V; i += blockDim.x) {
      ArgBest c = {x[i], i};
      best = arg_better(best, c);
    }
  }
  best = block_argmax(best, red_arg);
  if (!(T > 0.f)) {
    if (tid == 0) out[row] = best.i < 0 ? V - 1 : best.i;
    return;
  }
  const bool scale = T != 1.f;
  const float m = scale ? best.v / T : best.v;  // T > 0: the largest logit stays the largest

  // Each thread owns one contiguous chunk, so that prefix sums follow the index order.  Read straight from memory, long chunks
  // beside each other, every load of a wave would touch 64 lines, more than the caches of the compute unit keep; the
  // chunks therefore pass through LDS, DRAW_PART entries of each at a time, 32 neighbours a load (rows of 151,936 logits,
  // with filters in front: 205 us read straight, 94 so).  Short chunks are read as they lie (8 rows of 5,000: 16.6 us, through
  // LDS 24; of 16,384: 22 and 38; of 24,000: 40 straight, 39 through LDS, filtered 40 and 29).
  extern __shared__ float part[];            // [SAMPLE_THREADS][DRAW_PART + 1]
  const int per = (V + SAMPLE_THREADS - 1) / SAMPLE_THREADS;
  const int lo = min(V, tid * per), hi = min(V, lo + per);
  // (what the processors in front have dropped adds nothing; on the way through LDS a wave whose entries are all dropped skips the
  // arithmetic, which short chunks, whose loads are under way together, do not gain by)
  auto weight = [&](float v) { return expf((scale ? v / T : v) - m); };
  auto add_chunk = [&](float& sum, auto of) {
    if (per <= DRAW_DIRECT) {
#pragma unroll 8
      for (int i = lo; i < hi; ++i) sum += of(x[i]);
      return;
    }
    for (int at = 0; at < per; at += DRAW_PART) {
      __syncthreads();                       // (the part before has been read)
#pragma unroll
      for (int e = tid; e < SAMPLE_THREADS * DRAW_PART; e += SAMPLE_THREADS) {
        const int owner = e / DRAW_PART, k = at + e % DRAW_PART, i = owner * per + k;
        part[owner * (DRAW_PART + 1) + e % DRAW_PART] = k < per && i < V ? x[i] : 0.f;
      }
      __syncthreads();
      const int n = min(DRAW_PART, hi - lo - at);
      for (int k = 0; k < n; ++k) {
        const float v = part[tid * (DRAW_PART + 1) + k];
        if (v != -INFINITY) sum += of(v);
      }
    }
  };
  float s = 0.f;
  add_chunk(s, [&](float v) { return weight(v); });
  const float total = block_sum(s, red);
  float ps = 0.f;
  add_chunk(ps, [&](float v) { return weight(v) / total; });
  chunk_sum[tid] = ps;
  __syncthreads();
  // the sum of the chunks before this one, added one after another in their order: by every thread for itself, with long chunks
  // by one for all
  const int chunks = (V + per - 1) / per;
  float prefix = 0.f;
  if (per <= DRAW_DIRECT) {
    for (int t = 0; t < min(tid, chunks); ++t) prefix += chunk_sum[t];
  } else {
    if (tid == 0) {
      float sum = 0.f;
#pragma unroll 16
      for (int t = 0; t < chunks; ++t) {
        const float c = chunk_sum[t];
        chunk_sum[t] = sum;
        sum += c;
      }
    }
    __syncthreads();
    prefix = chunk_sum[tid];
  }
  const float u = uniform[row];
  int hit = V;  // none
  // A chunk whose end lies clearly below u has no hit (its entries added to `prefix` one by one and its own sum differ by no
  // more than the roundings of `per` additions below 2); those that begin above u come into question only if none before them has one.
  if (lo < hi && prefix <= u && u < prefix + ps + 2.4e-7f * (float)(per + 1)) {
    float c = prefix;
    for (int i0 = lo; i0 < hi && hit == V; i0 += 16) {
      float v[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) v[q] = i0 + q < hi ? x[i0 + q] : -INFINITY;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        if (hit == V && v[q] != -INFINITY) {      // (a dropped entry is never drawn, wherever the roundings of two chunks leave u)
          c += weight(v[q]) / total;
          if (u < c) hit = i0 + q;
        }
      }
    }
  }
  // the smallest (largest) of the threads' numbers, in all of them
  auto block_first = [&](int n, bool last) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int o = __shfl_xor(n, off, SYN_WAVE);
      n = last ? max(n, o) : min(n, o);
    }
    __syncthreads();
    if (tid % SYN_WAVE == 0) found[tid / SYN_WAVE] = n;
    __syncthreads();
    n = found[0];
    for (int w = 1; w < SAMPLE_THREADS / SYN_WAVE; ++w) n = last ? max(n, found[w]) : min(n, found[w]);
    return n;
  };
  int r = block_first(hit, false);
  if (r == V) {
    // u lies between two chunks: the first entry behind it that is not dropped.  Or nothing passes u (the rounded sum ends below it, or
    // is NaN): the last entry that is not dropped, of all of them the last.
    int first = V, last = -1;
    for (int i = lo; i < hi; ++i)
      if (x[i] != -INFINITY) last = i, first = min(first, i);
    r = block_first(prefix > u ? first : V, false);
    if (r == V) r = block_first(last, true);
    if (r < 0) r = V - 1;
  }
  if (tid == 0) out[row] = r;
}

SYN_EXPORT int syn_sample_rows(const float* logits, const float* temperature, const float* uniform, int* out,
                               int n_rows, int V, hipStream_t stream) {
  SYN_CHECK(n_rows > 0 && V > 0, "sample_rows: empty input (%d rows, vocabulary %d)", n_rows, V);
  SYN_CHECK(temperature == nullptr || uniform != nullptr, "sample_rows: temperatures need uniform numbers");
  const size_t lds = temperature && V > DRAW_DIRECT * SAMPLE_THREADS ? (size_t)SAMPLE_THREADS * (DRAW_PART + 1) * sizeof(float) : 0;     // (a draw's)
  static OncePerDevice raised;
  if (lds) {
    const hipError_t e = once_per_device(raised, [&] {
      return hipFuncSetAttribute((const void*)sample_rows_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    });
    SYN_CHECK(e == hipSuccess, "sample_rows: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
  }
  sample_rows_kernel<<<n_rows, SAMPLE_THREADS, lds, stream>>>(logits, temperature, uniform, out, V);
  SYN_LAUNCH_CHECK("sample_rows");
  return 0;
}

// ------------------------------------------------------------------ the processors in front of the sampler
// One workgroup a row of logits, in the reference's order (crates/synaptix-models/llm/common/src/generate.rs:304-340):
//   repetition penalty   once for each occurrence of a token in the row's list: a positive logit is divided,
//                        any other multiplied (crates/synaptix-infer/src/sampling/repetition.rs:27-45)
//   presence, frequency  logit -= presence + frequency * occurrences (repetition.rs:59-77)
//   temperature          logit /= T where T > 0 and T != 1 (logit_processor.rs:8-18)
//   top-k                the k largest stay (sampling/top_k.rs:8-24; of equal values at the k-th place the
//                        first in index order, where the reference's selection keeps arbitrary ones)
//   top-p                sorted by probability, a candidate stays while the sum of those before it is at most
//                        p * the sum of all (sampling/top_p.rs:8-44; equal probabilities in index order)
//   min-p                those below min_p * the largest probability go (sampling/min_p.rs:8-24)
// What is dropped becomes -inf.  The reference sorts on the host; here the k-th value and the boundary of the
// probability mass are found by selection on the float's bit pattern, a byte at a time from the top (four
// passes over the row with a histogram of 256 bins in LDS), and the sums are integers (probabilities in 44-bit
// fixed point), so that a row gives the same result whatever the order in which threads arrive.
#define FILTER_THREADS 1024
#define FILTER_LIST 2048
typedef unsigned long long u64;

// the float's bits as an unsigned number that grows with the float
__device__ __forceinline__ unsigned order_key(float x) {
  const unsigned b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ bool is_finite(float x) { return x > -INFINITY && x < INFINITY; }
__device__ __forceinline__ u64 mass_of(float x, float m) { return (u64)(expf(x - m) * 17592186044416.f); }   // * 2^44: up to 2^20 entries

struct FilterShared {
  unsigned cnt[256];
  u64 sum[256];
  u64 red64[FILTER_THREADS / SYN_WAVE];
  float redf[FILTER_THREADS / SYN_WAVE];
  int wave_n[FILTER_THREADS / SYN_WAVE];
  int bin;
  unsigned need;
  u64 above;
  // what top-k has left, if that is little: the processors behind it then walk this list, not the row
  int cand_j[FILTER_LIST];
  int n_cand;
};

__device__ __forceinline__ float block_max_all(float v, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, SYN_WAVE));
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = red[0];
#pragma unroll
  for (int i = 1; i < FILTER_THREADS / SYN_WAVE; ++i) t = fmaxf(t, red[i]);
  return t;
}
__device__ __forceinline__ u64 block_sum_all(u64 v, u64* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, SYN_WAVE);
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  u64 t = 0;
#pragma unroll
  for (int i = 0; i < FILTER_THREADS / SYN_WAVE; ++i) t += red[i];
  return t;
}

// For the lanes of one wave, lane l holding bins 4 l .. 4 l + 3 of a histogram: above[i] = the sum of all bins above
// bin 4 l + i.
template <typename T>
__device__ __forceinline__ void sums_above(const T* hist, int lane, T (&mine)[4], T (&above)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) mine[i] = hist[4 * lane + i];
  const T own = mine[0] + mine[1] + mine[2] + mine[3];
  T from_here = own;   // becomes the sum over this lane and all higher ones
#pragma unroll
  for (int off = 1; off < SYN_WAVE; off <<= 1) {
    const T o = __shfl_down(from_here, off, SYN_WAVE);
    if (lane + off < SYN_WAVE) from_here += o;
  }
  above[3] = from_here - own;
  above[2] = above[3] + mine[3];
  above[1] = above[2] + mine[2];
  above[0] = above[1] + mine[1];
}

// A thread's additions to the histogram go through one bin kept in registers: logits share their top bytes, and
// a thousand threads adding to the same few LDS words one by one would take longer than the pass itself.
struct BinCache {
  int bin = -1;
  unsigned n = 0;
  u64 s = 0;
  __device__ __forceinline__ void flush(FilterShared& sh, bool with_sums) {
    if (n) {
      atomicAdd(&sh.cnt[bin], n);
      if (with_sums) atomicAdd(&sh.sum[bin], s);
    }
    n = 0, s = 0;
  }
  __device__ __forceinline__ void add(FilterShared& sh, int b, u64 mass, bool with_sums) {
    if (b != bin) {
      flush(sh, with_sums);
      bin = b;
    }
    ++n, s += mass;
  }
};

// A pass over a row: f(j, x[j]) for every entry, 16 bytes a load and eight loads of a thread under way where the row
// allows it (one entry at a time, a pass of one workgroup over 150,000 entries waits 150 times for memory).
template <typename F>
__device__ __forceinline__ void for_each_entry(const float* x, int V, F f) {
  const int tid = threadIdx.x, nt = blockDim.x;
  if (V % 4 == 0 && (uintptr_t)x % 16 == 0) {
    const float4* x4 = (const float4*)x;
    const int V4 = V / 4;
    for (int i0 = tid; i0 < V4; i0 += 8 * nt) {
      float4 v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = i0 + q * nt < V4 ? x4[i0 + q * nt] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (i0 + q * nt < V4) {
          const int j = 4 * (i0 + q * nt);
          f(j, v[q].x), f(j + 1, v[q].y), f(j + 2, v[q].z), f(j + 3, v[q].w);
        }
    }
  } else {
    for (int j = tid; j < V; j += nt) f(j, x[j]);
  }
}
// The same with a new value for every entry: dst[j] = f(j, src[j]) (dst may be src).
template <typename F>
__device__ __forceinline__ void map_entries(const float* src, float* dst, int V, F f) {
  const int tid = threadIdx.x, nt = blockDim.x;
  if (V % 4 == 0 && (uintptr_t)src % 16 == 0 && (uintptr_t)dst % 16 == 0) {
    const float4* s4 = (const float4*)src;
    float4* d4 = (float4*)dst;
    const int V4 = V / 4;
    for (int i0 = tid; i0 < V4; i0 += 4 * nt) {
      float4 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = i0 + q * nt < V4 ? s4[i0 + q * nt] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (i0 + q * nt < V4) {
          const int j = 4 * (i0 + q * nt);
          d4[i0 + q * nt] = make_float4(f(j, v[q].x), f(j + 1, v[q].y), f(j + 2, v[q].z), f(j + 3, v[q].w));
        }
    }
  } else {
    for (int j = tid; j < V; j += nt) dst[j] = f(j, src[j]);
  }
}

// Of the entries whose key is `key`, those from the keep-th on in index order become -inf.
__device__ void drop_later_ties(float* x, int V, unsigned key, unsigned keep, FilterShared& sh) {
  const int tid = threadIdx.x, wave = tid / SYN_WAVE, lane = tid % SYN_WAVE, nw = blockDim.x / SYN_WAVE;
  unsigned before = 0;   // ties in earlier chunks; the same in every thread
  for (int base = 0; base < V; base += blockDim.x) {
    const int j = base + tid;
    const bool tie = j < V && order_key(x[j]) == key;
    const u64 votes = __ballot(tie);
    __syncthreads();
    if (lane == 0) sh.wave_n[wave] = __popcll(votes);
    __syncthreads();
    unsigned rank = before + __popcll(votes & ((1ull << lane) - 1ull)), all = 0;
    for (int w = 0; w < nw; ++w) {
      if (w < wave) rank += sh.wave_n[w];
      all += sh.wave_n[w];
    }
    if (tie && rank >= keep) x[j] = -INFINITY;
    before += all;
  }
  __syncthreads();
}

__global__ void __launch_bounds__(FILTER_THREADS)
filter_rows_kernel(const float* __restrict__ in, float* __restrict__ out, int V, const float* __restrict__ temperature,
                   const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ min_p,
                   const float* __restrict__ repetition, const float* __restrict__ presence,
                   const float* __restrict__ frequency, const int* __restrict__ ids, const int* __restrict__ id_start,
                   int* __restrict__ counts) {
  __shared__ FilterShared sh;
  const int row = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
  float* x = out + (size_t)row * V;
  const float* src = in + (size_t)row * V;    // the row as it comes, until the first pass that writes has copied it

  // ---- penalties: occurrences counted in the row's scratch counters, of which those of its tokens are zeroed before and after
  const int n_ids = id_start ? id_start[row + 1] - id_start[row] : 0;
  const float rep = repetition[row], pres = presence[row], freq = frequency[row];
  if (n_ids > 0 && (rep != 1.f || pres != 0.f || freq != 0.f)) {
    if (src != x) {
      map_entries(src, x, V, [](int, float v) { return v; });
      src = x;
      __syncthreads();
    }
    int* cnt = counts + (size_t)row * V;
    const int* mine = ids + id_start[row];
    for (int i = tid; i < n_ids; i += nt) {
      const int t = mine[i];
      if (t >= 0 && t < V) cnt[t] = 0;
    }
    __syncthreads();
    for (int i = tid; i < n_ids; i += nt) {
      const int t = mine[i];
      if (t >= 0 && t < V) atomicAdd(&cnt[t], 1);
    }
    __syncthreads();
    for (int i = tid; i < n_ids; i += nt) {
      const int t = mine[i];
      if (t < 0 || t >= V) continue;
      const int c = __hip_atomic_load(&cnt[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (c > 0 && atomicCAS(&cnt[t], c, -c) == c) {   // one of the token's occurrences does the work
        float v = x[t];
        if (rep != 1.f) {
          const float f = powf(rep, (float)c);
          v = v > 0.f ? v / f : v * f;
        }
        if (pres != 0.f || freq != 0.f) v -= pres + freq * (float)c;
        x[t] = v;
      }
    }
    __syncthreads();
    for (int i = tid; i < n_ids; i += nt) {
      const int t = mine[i];
      if (t >= 0 && t < V) cnt[t] = 0;
    }
    __syncthreads();
  }

  // ---- temperature, and the largest logit (which every later step keeps); with top-k the histogram of the top byte as well
  const float T = temperature[row];
  const bool scale = T > 0.f && T != 1.f;
  const int k = top_k[row];
  const bool cut = k > 0 && k < V;
  if (cut) {
    for (int b = tid; b < 256; b += nt) sh.cnt[b] = 0;
    if (tid == 0) sh.n_cand = 0;
    __syncthreads();
  }
  float m = -INFINITY;
  auto first_pass = [&](auto with_histogram) {      // (two loops: rows without top-k pay nothing for it)
    BinCache top;
    auto seen = [&](float v) {
      m = fmaxf(m, v);
      if constexpr (decltype(with_histogram)::value) top.add(sh, order_key(v) >> 24, 0, false);
    };
    if (scale || src != x) {
      map_entries(src, x, V, [&](int, float v) {
        if (scale) v = v / T;
        seen(v);
        return v;
      });
    } else {
      for_each_entry(x, V, [&](int, float v) { seen(v); });
    }
    if constexpr (decltype(with_histogram)::value) top.flush(sh, false);
  };
  if (cut) first_pass(std::true_type{});
  else first_pass(std::false_type{});
  m = block_max_all(m, sh.redf);   // (its barriers also stand between the writes above and the reads below)

  // ---- top-k: the key of the k-th largest, a byte at a time.  Once few enough entries can still be among the k (after two
  // bytes, with logits as they come, some hundreds), one pass lists them in LDS (in no order) and drops the others: a
  // row is walked three times (151,936 logits: about 15 us a pass) instead of six.
  bool listed = false;
  if (cut) {
    unsigned prefix = 0, need = (unsigned)k, ties = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
      const unsigned himask = shift == 24 ? 0u : 0xffffffffu << (shift + 8);
      if (shift < 24) {
        for (int b = tid; b < 256; b += nt) sh.cnt[b] = 0;
        __syncthreads();
        BinCache cache;
        auto count = [&](int, float v) {
          const unsigned key = order_key(v);
          if ((key & himask) == prefix) cache.add(sh, (key >> shift) & 255, 0, false);
        };
        if (listed) {
          for (int i = tid; i < sh.n_cand; i += nt) count(0, x[sh.cand_j[i]]);
        } else {
          for_each_entry(x, V, count);
        }
        cache.flush(sh, false);
        __syncthreads();
      }
      if (tid < SYN_WAVE) {
        // the bin in which the need-th largest of the matching entries lies (there are at least `need` of them)
        unsigned mine[4], above[4];
        sums_above(sh.cnt, tid, mine, above);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (above[i] < need && need <= above[i] + mine[i]) sh.bin = 4 * tid + i, sh.need = need - above[i];
      }
      __syncthreads();
      prefix |= (unsigned)sh.bin << shift, need = sh.need, ties = sh.cnt[sh.bin];
      __syncthreads();
      // above the prefix lie k - need entries, `ties` share it (all the same in every thread)
      if (!listed && shift > 0 && shift < 24 && (unsigned)k - need + ties <= FILTER_LIST) {
        map_entries(x, x, V, [&](int j, float v) {
          if (order_key(v) < prefix) return -INFINITY;
          sh.cand_j[atomicAdd(&sh.n_cand, 1)] = j;
          return v;
        });
        __syncthreads();
        listed = true;
      }
    }
    // below the k-th key everything goes; of its equals the first `need` stay.  What stays is listed for the processors behind.
    if (listed) {
      for (int i = tid; i < sh.n_cand; i += nt)
        if (order_key(x[sh.cand_j[i]]) < prefix) x[sh.cand_j[i]] = -INFINITY;
    } else {
      const bool list = (unsigned)k - need + ties <= FILTER_LIST;
      map_entries(x, x, V, [&](int j, float v) {
        if (order_key(v) < prefix) return -INFINITY;
        if (list) sh.cand_j[atomicAdd(&sh.n_cand, 1)] = j;
        return v;
      });
      listed = list;
    }
    __syncthreads();
    if (need < ties) drop_later_ties(x, V, prefix, need, sh);
  }
  // a pass over what is left: f(j, value) for the listed entries or for the whole row
  const int n_listed = listed ? sh.n_cand : 0;
  auto each_left = [&](auto f) {
    if (listed) {
      for (int i = tid; i < n_listed; i += nt) f(sh.cand_j[i], x[sh.cand_j[i]]);
    } else {
      for_each_entry(x, V, f);
    }
  };
  auto drop_left = [&](auto gone) {   // gone(value): whether the entry goes
    if (listed) {
      for (int i = tid; i < n_listed; i += nt) {
        const int j = sh.cand_j[i];
        if (gone(x[j])) x[j] = -INFINITY;
      }
    } else {
      map_entries(x, x, V, [&](int, float v) { return gone(v) ? -INFINITY : v; });
    }
  };

  // ---- top-p: the lowest key whose mass above it is at most p * all mass
  const float p = top_p[row], mp = min_p[row];
  bool min_p_done = false;
  if (p < 1.f) {
    u64 limit = 0;       // p * all mass; all mass is what the first histogram adds up to
    unsigned prefix = 0, ties = 0;
    u64 above = 0, tie_mass = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
      const unsigned himask = shift == 24 ? 0u : 0xffffffffu << (shift + 8);
      for (int b = tid; b < 256; b += nt) sh.cnt[b] = 0, sh.sum[b] = 0;
      __syncthreads();
      BinCache cache;
      each_left([&](int, float v) {
        if (!is_finite(v)) return;
        const unsigned key = order_key(v);
        if ((key & himask) == prefix) cache.add(sh, (key >> shift) & 255, mass_of(v, m), true);
      });
      cache.flush(sh, true);
      __syncthreads();
      if (tid < SYN_WAVE) {
        // a bin's largest entry has exactly the mass of the bins above it before it: the lowest bin that holds
        // entries and has at most `limit` above it is where the boundary lies (every such bin above it stays whole)
        u64 mine[4], over[4];
        sums_above(sh.sum, tid, mine, over);
        if (shift == 24) {
          const u64 total = __shfl(over[0] + mine[0], 0, SYN_WAVE);
          limit = (u64)((double)p * (double)total);
          if (tid == 0) sh.red64[0] = limit;
        }
        int lowest = 256;
#pragma unroll
        for (int i = 3; i >= 0; --i)
          if (sh.cnt[4 * tid + i] && above + over[i] <= limit) lowest = 4 * tid + i;
        int first = lowest;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) first = min(first, __shfl_xor(first, off, SYN_WAVE));
        if (first == 256) {
          if (tid == 0) sh.bin = -1;
        } else if (first == lowest) {
          sh.bin = first, sh.above = above + over[first % 4];
        }
      }
      __syncthreads();
      if (sh.bin < 0) break;   // no finite entry at all
      limit = sh.red64[0];
      prefix |= (unsigned)sh.bin << shift, above = sh.above, ties = sh.cnt[sh.bin], tie_mass = sh.sum[sh.bin];
      __syncthreads();
    }
    if (ties > 0) {
      // (min-p looks at each entry alone, so it goes along in this pass)
      drop_left([&](float v) { return is_finite(v) && (order_key(v) < prefix || (mp > 0.f && expf(v - m) < mp)); });
      min_p_done = true;
      __syncthreads();
      // the j-th of equal entries has (j - 1) of them before it as well
      const u64 each = tie_mass / ties;
      const u64 keep = each == 0 ? (u64)ties : (limit - above) / each + 1;
      if (keep < ties) drop_later_ties(x, V, prefix, (unsigned)keep, sh);
    }
  }

  // ---- min-p: the largest probability belongs to the largest logit, exp(0) = 1 before the division by the sum
  if (mp > 0.f && !min_p_done) drop_left([&](float v) { return is_finite(v) && expf(v - m) < mp; });
}

// in, out [n_rows, V] float (may be the same); one entry a row of every option (top_k 0 and top_p >= 1: off);
// ids, id_start [n_rows + 1]: the tokens that the penalties look at, row after row (null: none);
// counts [n_rows * V] int, any content: this call's own (needed with ids)
SYN_EXPORT int syn_filter_rows(const float* in, float* out, int n_rows, int V, const float* temperature, const int* top_k,
                               const float* top_p, const float* min_p, const float* repetition, const float* presence,
                               const float* frequency, const int* ids, const int* id_start, int* counts,
                               hipStream_t stream) {
  SYN_CHECK(n_rows > 0 && V > 0 && V <= (1 << 20), "filter_rows: %d rows, vocabulary %d (1 .. 2^20)", n_rows, V);
  SYN_CHECK(in && out && temperature && top_k && top_p && min_p && repetition && presence && frequency,
            "filter_rows: an option array is missing");
  SYN_CHECK((ids == nullptr) == (id_start == nullptr) && (ids == nullptr || counts != nullptr),
            "filter_rows: the penalties' tokens come with their row offsets and with counters");
  filter_rows_kernel<<<n_rows, FILTER_THREADS, 0, stream>>>(in, out, V, temperature, top_k, top_p, min_p, repetition,
                                                            presence, frequency, ids, id_start, counts);
  SYN_LAUNCH_CHECK("filter_rows");
  return 0;
}

// ------------------------------------------------------------------ filters and draw of rows with a top-k, many workgroups a row
// With a top-k the processors keep few entries, and a token can be drawn from those alone: no row is written, and the row is
// read once, by as many workgroups as it has slices.  What bounds it: the start of two kernels and the walk of a slice of some
// thousand entries through LDS, then of the slices' candidates by one workgroup.
//   1  topk_slices: a workgroup takes a slice of the row into LDS, applies the penalties (their tokens counted in LDS) and the
//      temperature, finds the slice's own k largest and stores them in index order;
//   2  topk_draw: a workgroup a row finds the k largest of these, which are the row's (of equal values the first in index order:
//      the slices and what they store lie in that order), then top-p, min-p and the draw on the at most TOPK_MAX that are left.
// Every step takes the same roundings in the same order as the kernels above (the sums of top-p are whole numbers, those of the
// draw go chunk by chunk as there), so a row's token is the one that they give.  8 rows of 151,936 logits with penalties,
// top-k 50 and top-p: 104 + 95 us as two kernels of a workgroup a row, 18 + 19 so; a call with its upload and the token's way back
// 305 -> 150 us.
#define TOPK_MAX 512         // of a row's k; with TOPK_SLICES slices their candidates fill 128 KB of LDS
#define TOPK_SLICES 32
#define TOPK_SLICE_MAX 8192  // entries of a slice: 32 KB of values and as much for the counters
#define SLICE_THREADS 512

template <int NT>
struct SelectShared {
  unsigned hist[2048];
  unsigned wave_n[2][NT / SYN_WAVE];
  unsigned bin, need, ties;
};

// Of the n keys that `key` returns those above `prefix` and the first `need` that equal it are the k largest (1 <= k <= n): 11, 11
// and 10 bits of the keys at a time from the top, with a histogram each.
template <int NT, typename F>
__device__ __forceinline__ void kth_key(F key, int n, unsigned k, SelectShared<NT>& sh, unsigned& prefix, unsigned& need) {
  constexpr int BINS = 2048 / NT;
  const int tid = threadIdx.x, wave = tid / SYN_WAVE, lane = tid % SYN_WAVE;
  unsigned ties;
  prefix = 0, need = k;
  for (int pass = 0; pass < 3; ++pass) {
    const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0;
    const unsigned low = pass == 2 ? 1023u : 2047u, himask = pass == 0 ? 0u : pass == 1 ? 0xffe00000u : 0xfffffc00u;
    for (int b = tid; b < 2048; b += NT) sh.hist[b] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += NT) {
      const unsigned q = key(i);
      if ((q & himask) == prefix) atomicAdd(&sh.hist[(q >> shift) & low], 1u);
    }
    __syncthreads();
    unsigned mine[BINS], own = 0;
#pragma unroll
    for (int i = 0; i < BINS; ++i) mine[i] = sh.hist[BINS * tid + i], own += mine[i];
    unsigned from_here = own;       // becomes the sum over this lane's bins and those of all higher lanes
#pragma unroll
    for (int off = 1; off < SYN_WAVE; off <<= 1) {
      const unsigned o = __shfl_down(from_here, off, SYN_WAVE);
      if (lane + off < SYN_WAVE) from_here += o;
    }
    if (lane == 0) sh.wave_n[0][wave] = from_here;
    __syncthreads();
    unsigned above = from_here - own;
#pragma unroll
    for (int w = 0; w < NT / SYN_WAVE; ++w) above += w > wave ? sh.wave_n[0][w] : 0u;
#pragma unroll
    for (int i = BINS - 1; i >= 0; --i) {
      if (above < need && need <= above + mine[i]) sh.bin = BINS * tid + i, sh.need = need - above, sh.ties = mine[i];
      above += mine[i];
    }
    __syncthreads();
    prefix |= sh.bin << shift, need = sh.need, ties = sh.ties;
    __syncthreads();
    if (need == ties && prefix > 0) {      // everything from here up belongs to them: no need to look at the bits below
      --prefix, need = 0;
      return;
    }
  }
}

// put(i, place) for the entries i < n above `prefix` and the first `need` that equal it, in index order; returns how many.  Each wave
// takes a run of neighbours, counts what is in it, and places them behind those of the waves before it.
template <int NT, typename F, typename G>
__device__ __forceinline__ int keep_largest(F key, int n, unsigned prefix, unsigned need, SelectShared<NT>& sh, G put) {
  constexpr int NW = NT / SYN_WAVE;
  const int wave = threadIdx.x / SYN_WAVE, lane = threadIdx.x % SYN_WAVE;
  const int run = (n + NT - 1) / NT * SYN_WAVE, lo = wave * run, hi = min(n, lo + run);
  const u64 below = (1ull << lane) - 1ull;
  unsigned more_n = 0, ties_n = 0;
  for (int i0 = lo; i0 < hi; i0 += SYN_WAVE) {
    const int i = i0 + lane;
    const unsigned q = i < hi ? key(i) : 0u;
    more_n += __popcll(__ballot(i < hi && q > prefix));
    ties_n += __popcll(__ballot(i < hi && q == prefix));
  }
  if (lane == 0) sh.wave_n[0][wave] = ties_n, sh.wave_n[1][wave] = more_n;
  __syncthreads();
  unsigned ties = 0, more = 0, ties_all = 0, more_all = 0;      // in front of this wave's run; everywhere
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const unsigned t = sh.wave_n[0][w], m = sh.wave_n[1][w];
    if (w < wave) ties += t, more += m;
    ties_all += t, more_all += m;
  }
  if (more_n + ties_n > 0) {
    for (int i0 = lo; i0 < hi; i0 += SYN_WAVE) {
      const int i = i0 + lane;
      const unsigned q = i < hi ? key(i) : 0u;
      const bool is_more = i < hi && q > prefix, is_tie = i < hi && q == prefix;
      const u64 v_more = __ballot(is_more), v_tie = __ballot(is_tie);
      const unsigned ties_at = ties + __popcll(v_tie & below);
      // (in front of an entry stay the larger ones, and of its equals no more than `need`)
      if (is_more || (is_tie && ties_at < need)) put(i, (int)(more + __popcll(v_more & below) + min(ties_at, need)));
      more += __popcll(v_more), ties += __popcll(v_tie);
    }
  }
  return (int)(more_all + min(ties_all, need));
}

__global__ void __launch_bounds__(SLICE_THREADS)
topk_slices_kernel(const float* __restrict__ in, int V, int slice, const float* __restrict__ temperature,
                   const int* __restrict__ top_k, const float* __restrict__ repetition, const float* __restrict__ presence,
                   const float* __restrict__ frequency, const int* __restrict__ ids, const int* __restrict__ id_start,
                   float* __restrict__ cand_v, int* __restrict__ cand_i, int* __restrict__ cand_n) {
  __shared__ SelectShared<SLICE_THREADS> sh;
  extern __shared__ __align__(16) float val[];   // [slice], and behind them the counters [slice]
  int* cnt = (int*)(val + slice);
  const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
  const int lo = part * slice, n = min(slice, V - lo);
  const float* x = in + (size_t)row * V + lo;
  if (V % 4 == 0 && (uintptr_t)in % 16 == 0) {   // (a slice is a multiple of four entries)
    const float4* x4 = (const float4*)x;
    float4* d4 = (float4*)val;
    const int n4 = n / 4;
    for (int i0 = tid; i0 < n4; i0 += 4 * SLICE_THREADS) {
      float4 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (i0 + q * SLICE_THREADS < n4) v[q] = x4[i0 + q * SLICE_THREADS];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (i0 + q * SLICE_THREADS < n4) d4[i0 + q * SLICE_THREADS] = v[q];
    }
  } else {
    for (int j = tid; j < n; j += SLICE_THREADS) val[j] = x[j];
  }
  const int first = id_start ? id_start[row] : 0, n_ids = id_start ? id_start[row + 1] - first : 0;
  const float rep = repetition[row], pres = presence[row], freq = frequency[row];
  const bool penalties = n_ids > 0 && (rep != 1.f || pres != 0.f || freq != 0.f);
  if (penalties) {
    for (int j = tid; j < n; j += SLICE_THREADS) cnt[j] = 0;
    __syncthreads();
    for (int i = tid; i < n_ids; i += SLICE_THREADS) {
      const int t = ids[first + i];
      if (t >= lo && t < lo + n) atomicAdd(&cnt[t - lo], 1);
    }
  }
  __syncthreads();
  const float T = temperature[row];
  const bool scale = T > 0.f && T != 1.f;
  if (penalties || scale) {
    for (int j = tid; j < n; j += SLICE_THREADS) {
      float v = val[j];
      const int c = penalties ? cnt[j] : 0;
      if (c > 0) {
        if (rep != 1.f) {
          const float f = powf(rep, (float)c);
          v = v > 0.f ? v / f : v * f;
        }
        if (pres != 0.f || freq != 0.f) v -= pres + freq * (float)c;
      }
      val[j] = scale ? v / T : v;
    }
    __syncthreads();
  }
  const int k = max(1, min(top_k[row], TOPK_MAX));
  auto key = [&](int i) { return order_key(val[i]); };
  unsigned prefix = 0, need = 0;
  if (k < n) kth_key<SLICE_THREADS>(key, n, (unsigned)k, sh, prefix, need);      // (else prefix 0: all of them stay)
  const size_t at = ((size_t)row * gridDim.x + part) * TOPK_MAX;
  const int kept = keep_largest<SLICE_THREADS>(key, n, prefix, k < n ? need : (unsigned)n, sh, [&](int i, int place) {
    cand_v[at + place] = val[i];
    cand_i[at + place] = lo + i;
  });
  if (tid == 0) cand_n[row * gridDim.x + part] = kept;
}

__global__ void __launch_bounds__(SAMPLE_THREADS)
topk_draw_kernel(const float* __restrict__ cand_v, const int* __restrict__ cand_i, const int* __restrict__ cand_n, int parts,
                 int V, const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ min_p,
                 const float* __restrict__ draw, const float* __restrict__ uniform, int* __restrict__ out) {
  __shared__ SelectShared<SAMPLE_THREADS> sh;
  __shared__ float kept_v[TOPK_MAX], chunk_at[TOPK_MAX];
  __shared__ int kept_i[TOPK_MAX];
  __shared__ u64 mass[TOPK_MAX];
  __shared__ unsigned keys[TOPK_MAX];
  __shared__ u64 red64[SAMPLE_THREADS / SYN_WAVE];
  __shared__ float redf[SAMPLE_THREADS / SYN_WAVE];
  __shared__ ArgBest red_arg[SAMPLE_THREADS / SYN_WAVE];
  __shared__ float chunk_sum[SAMPLE_THREADS];
  __shared__ int starts[TOPK_SLICES + 1];
  __shared__ int found[2];
  extern __shared__ float all_v[];               // [parts * TOPK_MAX] values, and behind them their places in the row
  int* all_i = (int*)(all_v + parts * TOPK_MAX);
  const int row = blockIdx.x, tid = threadIdx.x;

  if (tid < SYN_WAVE) {
    int n = tid < parts ? cand_n[row * parts + tid] : 0;
    const int own = n;
#pragma unroll
    for (int off = 1; off < TOPK_SLICES; off <<= 1) {
      const int o = __shfl_up(n, off, SYN_WAVE);
      if (tid >= off) n += o;
    }
    if (tid < parts) starts[tid] = n - own;
    if (tid == parts - 1) starts[parts] = n;
  }
  __syncthreads();
  const int n_all = starts[parts];
  for (int p = tid / SYN_WAVE; p < parts; p += SAMPLE_THREADS / SYN_WAVE) {
    const size_t at = ((size_t)row * parts + p) * TOPK_MAX;
    for (int i = tid % SYN_WAVE; i < starts[p + 1] - starts[p]; i += SYN_WAVE)
      all_v[starts[p] + i] = cand_v[at + i], all_i[starts[p] + i] = cand_i[at + i];
  }
  __syncthreads();

  // ---- top-k
  // (k < V and a slice has left out entries only if it kept k, so there are k of them)
  const unsigned k = (unsigned)max(1, min(min(top_k[row], TOPK_MAX), n_all));
  unsigned prefix, need;
  auto key = [&](int i) { return order_key(all_v[i]); };
  kth_key<SAMPLE_THREADS>(key, n_all, k, sh, prefix, need);
  const int n = keep_largest<SAMPLE_THREADS>(key, n_all, prefix, need, sh, [&](int i, int place) {
    kept_v[place] = all_v[i], kept_i[place] = all_i[i];
  });
  __syncthreads();

  // ---- top-p and min-p, an entry a thread: an entry stays while the mass of those before it (larger, or equal and earlier) is
  // at most p * all mass, which is what the radix search above finds the boundary of
  const float p = top_p[row], mp = min_p[row];
  float mine = tid < n ? kept_v[tid] : -INFINITY;
  const float m = block_max_all(mine, redf);
  if (p < 1.f) {
    const bool counts = tid < n && is_finite(mine);
    const u64 own = counts ? mass_of(mine, m) : 0;
    const unsigned mk = order_key(mine);
    if (tid < n) mass[tid] = own, keys[tid] = mk;
    const u64 total = block_sum_all(own, red64);
    const u64 limit = (u64)((double)p * (double)total);
    if (counts) {
      u64 before = 0;
#pragma unroll 8
      for (int j = 0; j < n; ++j) {
        const unsigned q = keys[j];
        const u64 w = mass[j];
        before += (q > mk) | ((q == mk) & (j < tid)) ? w : 0;
      }
      if (before > limit) mine = -INFINITY;
    }
  }
  if (mp > 0.f && is_finite(mine) && expf(mine - m) < mp) mine = -INFINITY;
  __syncthreads();
  if (tid < n) kept_v[tid] = mine;
  if (tid < 2) found[tid] = tid == 0 ? V : -1;
  chunk_sum[tid] = 0.f;
  // (a NaN is larger than nothing; the barriers inside end the writes above)
  const ArgBest best = block_argmax(arg_better(ArgBest{-INFINITY, -1}, ArgBest{mine, tid < n ? kept_i[tid] : -1}), red_arg);

  if (!(draw[row] > 0.f)) {
    if (tid == 0) {
      int r = best.i;
      if (!(best.v > -INFINITY)) {     // nothing is larger than -inf: the last entry that is -inf, among all entries of the row
        r = V - 1;
        for (int j = n - 1; j >= 0 && kept_i[j] == r && kept_v[j] != -INFINITY; --j) --r;
        if (r < 0) r = V - 1;
      }
      out[row] = r;
    }
    return;
  }

  // ---- the draw, as sample_rows takes it at temperature 1: chunks of the row, each by the thread of its first entry
  const float top = best.v;
  const int per = (V + SAMPLE_THREADS - 1) / SAMPLE_THREADS;
  const int chunk = tid < n ? kept_i[tid] / per : -1;
  const bool opens = tid < n && (tid == 0 || kept_i[tid - 1] / per != chunk);
  int end = tid;
  if (opens) {
    float s = 0.f;
    for (; end < n && kept_i[end] / per == chunk; ++end)
      if (kept_v[end] != -INFINITY) s += expf(kept_v[end] - top);
    chunk_sum[chunk] = s;
  }
  __syncthreads();
  const float total = block_sum(chunk_sum[tid], redf);
  float ps = 0.f;
  if (opens)
    for (int j = tid; j < end; ++j)
      if (kept_v[j] != -INFINITY) ps += expf(kept_v[j] - top) / total;
  if (tid < n) chunk_at[tid] = opens ? ps : 0.f;
  __syncthreads();
  if (tid == 0) {
    float sum = 0.f;      // (chunks without entries add nothing)
    for (int j0 = 0; j0 < n; j0 += 16) {
      float c[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) c[q] = j0 + q < n ? chunk_at[j0 + q] : 0.f;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        if (j0 + q < n) chunk_at[j0 + q] = sum;
        sum += c[q];
      }
    }
  }
  __syncthreads();
  const float u = uniform[row];
  const float before = opens ? chunk_at[tid] : 0.f;
  if (opens && before <= u && u < before + ps + 2.4e-7f * (float)(per + 1)) {
    float c = before;
    for (int j = tid; j < end; ++j)
      if (kept_v[j] != -INFINITY) {
        c += expf(kept_v[j] - top) / total;
        if (u < c) {
          atomicMin(&found[0], kept_i[j]);
          break;
        }
      }
  }
  __syncthreads();
  int r = found[0];
  if (r == V) {
    // as in sample_rows: the first entry that is left in a chunk behind u, else the last one that is left
    __syncthreads();
    if (opens)
      for (int j = tid; j < end; ++j)
        if (kept_v[j] != -INFINITY) {
          if (before > u) atomicMin(&found[0], kept_i[j]);
          atomicMax(&found[1], kept_i[j]);
        }
    __syncthreads();
    r = found[0] < V ? found[0] : found[1] >= 0 ? found[1] : V - 1;
  }
  if (tid == 0) out[row] = r;
}

// Slices of a row: as many as the chip has room for at few rows, of at least 1,024 entries.
static int topk_slice(int V) {
  const int parts = V / 1024 < 1 ? 1 : V / 1024 > TOPK_SLICES ? TOPK_SLICES : V / 1024;
  return ((V + parts - 1) / parts + 3) / 4 * 4;
}
// Four-byte words of scratch memory that syn_draw_top_k needs for n_rows rows of V logits; 0: it does not take rows of this size.
SYN_EXPORT long syn_draw_top_k_words(int n_rows, int V) {
  const int slice = V > 0 ? topk_slice(V) : 0;
  if (n_rows <= 0 || n_rows > 65535 || V <= 0 || slice > TOPK_SLICE_MAX) return 0;
  return (long)n_rows * ((V + slice - 1) / slice) * (2 * TOPK_MAX + 1);
}

// filter_rows and sample_rows in one for rows that all have a top-k (1 <= top_k <= TOPK_MAX, top_k < V; the rows' largest is max_k):
// the token of every row to out.  draw: greedy where <= 0, else the row is drawn from with `uniform`.  words: syn_draw_top_k_words of
// scratch memory with any content.
SYN_EXPORT int syn_draw_top_k(const float* logits, int n_rows, int V, int max_k, const float* temperature, const int* top_k,
                              const float* top_p, const float* min_p, const float* repetition, const float* presence,
                              const float* frequency, const int* ids, const int* id_start, const float* draw,
                              const float* uniform, float* words, int* out, hipStream_t stream) {
  SYN_CHECK(syn_draw_top_k_words(n_rows, V) > 0, "draw_top_k: %d rows of %d logits", n_rows, V);
  SYN_CHECK(logits && temperature && top_k && top_p && min_p && repetition && presence && frequency && draw && uniform && words && out,
            "draw_top_k: an array is missing");
  SYN_CHECK((ids == nullptr) == (id_start == nullptr), "draw_top_k: the penalties' tokens come with their row offsets");
  SYN_CHECK(max_k >= 1 && max_k <= TOPK_MAX && max_k < V, "draw_top_k: top-k up to %d of %d logits (at most %d)", max_k, V, TOPK_MAX);
  const int slice = topk_slice(V), parts = (V + slice - 1) / slice;
  const size_t lds_slice = (size_t)slice * 8, lds_draw = (size_t)parts * TOPK_MAX * 8;
  static OncePerDevice raised;
  const hipError_t e = once_per_device(raised, [&] {
    const hipError_t a = hipFuncSetAttribute((const void*)topk_slices_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             TOPK_SLICE_MAX * 8);
    return a != hipSuccess ? a : hipFuncSetAttribute((const void*)topk_draw_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     TOPK_SLICES * TOPK_MAX * 8);
  });
  SYN_CHECK(e == hipSuccess, "draw_top_k: %zu and %zu bytes of LDS refused: %s", lds_slice, lds_draw, hipGetErrorString(e));
  const size_t n_cand = (size_t)n_rows * parts * TOPK_MAX;
  int* cand_i = (int*)(words + n_cand);
  int* cand_n = (int*)(words + 2 * n_cand);
  topk_slices_kernel<<<dim3(parts, n_rows), SLICE_THREADS, lds_slice, stream>>>(logits, V, slice, temperature, top_k, repetition,
                                                                               presence, frequency, ids, id_start, words, cand_i, cand_n);
  SYN_LAUNCH_CHECK("draw_top_k");
  topk_draw_kernel<<<n_rows, SAMPLE_THREADS, lds_draw, stream>>>(words, cand_i, cand_n, parts, V, top_k, top_p, min_p, draw, uniform, out);
  SYN_LAUNCH_CHECK("draw_top_k");
  return 0;
}
