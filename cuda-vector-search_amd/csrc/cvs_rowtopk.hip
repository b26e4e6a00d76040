// Exact top-k of each row of an fp32 score matrix, k <= 1024 (the large-k path,
// which the reference leaves to torch.topk: index.py:118, reference.py:8-15).
//
// Bound by reading the matrix (4 bytes per score, out of the 256 MB MALL while
// it fits), so a row's scores are read once, by as many workgroups as fill the
// GPU, and all further work is on the ~1.5k scores above a sampled threshold:
//
//  1. row_sample_kernel, one workgroup per row: a threshold that some 1.2k..3k
//     of the row's scores should reach, from a sample of 128-byte groups spread
//     evenly over the row (even a corpus stored topic by topic is sampled in
//     proportion);
//  2. row_filter_kernel, one workgroup per (row, chunk): the scores at or above
//     the threshold into the row's candidate array;
//  3. row_final_kernel, one workgroup per row: cuts the candidates to few more
//     than k, ranks those and writes the k best.  The threshold is a guess and never decides the result: when
//     fewer than k or more than kRowCap scores reach it, the row is streamed
//     again here and its top k taken exactly.
//
// Rows of at most kRowDirect scores need no threshold: step 3 takes the whole row.
// With two or more rows a CU, one workgroup of 256 threads does a long row's three
// steps (kStream), the candidates in LDS.
//
// Measured against chunk-wise radix selects and a merge of the chunks' top k:
// 64 rows x 300k, k = 1000: 189 -> 49 us; 1 x 4M, k = 1000: 3380 -> 60 us; whole
// rows, 1000 x 8000, k = 1000: 77 -> 46 us; 4000 x 40000, k = 100: 258 -> 188.
#include "cvs_common.h"
#include "cvs_kernels.h"

namespace cvs {

namespace {

// T below: threads of a row's workgroup, 1024, or 256 and 512 where there are
// several rows a CU (barriers then wait for fewer waves, and 7 or 4 rows share a CU).
constexpr int kNarrow = 256;
constexpr int kBins = 1024;
constexpr int kFilterU = 16;              // scores per thread and round of the filter
constexpr int kFilterFlush = 512;         // candidates in LDS that trigger a write-out
constexpr int kFilterRound = kBlock * kFilterU;

// Linear bins over [lo, hi], non-decreasing in the score, in [0, kBins) for
// any score (NaN: bin 0).
struct Bins {
  float lo, scale;
  __device__ __forceinline__ int of(float v) const {
    const float t = (v - lo) * scale;
    return (int)(t >= 0.f ? fminf(t, (float)(kBins - 1)) : 0.f);
  }
};

template <int T>
struct BinScratch {
  float mm[2][T / kWave];
  int hist[kBins];
  int wsum[T / kWave];
  int bin, above;
};

// The block's bins over the [min, max] of every thread's (lo, hi), an empty
// histogram, and false when that range is empty or not finite.  Whole block.
template <int T>
__device__ __forceinline__ bool make_bins(BinScratch<T>& B, float lo, float hi, Bins* bins) {
  const int tid = threadIdx.x;
  lo = wave_min_f32(lo);
  hi = wave_max_f32(hi);
  if (tid % kWave == 0) {
    B.mm[0][tid / kWave] = lo;
    B.mm[1][tid / kWave] = hi;
  }
#pragma unroll
  for (int i = 0; i < kBins / T; ++i) B.hist[i * T + tid] = 0;
  __syncthreads();
  lo = B.mm[0][0];
  hi = B.mm[1][0];
#pragma unroll
  for (int i = 1; i < T / kWave; ++i) {
    lo = fminf(lo, B.mm[0][i]);
    hi = fmaxf(hi, B.mm[1][i]);
  }
  const float width = hi - lo;
  bins->lo = lo;
  bins->scale = (float)kBins / width;
  return width > 0.f && __builtin_isfinite(width) && __builtin_isfinite(bins->scale);
}

// The highest bin b with at least `want` counts in bins >= b (bin 0 when there
// are fewer in all), and that count.  Whole block, after a barrier that made
// the histogram complete.
template <int T>
__device__ __forceinline__ int cut_bin(BinScratch<T>& B, int want, int* above) {
  constexpr int Q = kBins / T;  // bins a thread, descending
  const int tid = threadIdx.x;
  int c[Q], sum = 0;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    c[i] = B.hist[kBins - 1 - tid * Q - i];
    sum += c[i];
  }
  int incl = wave_incl_sum_i32(sum);
  if (tid % kWave == kWave - 1) B.wsum[tid / kWave] = incl;
  if (tid == 0) B.bin = -1;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < T / kWave; ++w) incl += w < tid / kWave ? B.wsum[w] : 0;
  int run = incl - sum;
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    if (run < want && want <= run + c[i]) {
      B.bin = kBins - 1 - tid * Q - i;
      B.above = run + c[i];
    }
    run += c[i];
  }
  __syncthreads();
  *above = B.above;
  return B.bin;
}

// A set {v >= floor, bins.of(v) >= bin} that holds the k best of a block's values.
struct Cut {
  Bins bins;
  float floor;
  int bin;
  __device__ __forceinline__ bool keeps(float v) const { return v >= floor && bins.of(v) >= bin; }  // (no NaN)
};

// A cut of at most `want` values where there is one: linear bins over the values'
// range, then over the range of the values in the bin that holds the k-th best,
// as long as that one holds too many (a few large values leave all others in
// one bin).  Returns the count of the cut, kNoCut without one (fewer than k
// values, all equal).  each(f) calls f(v) for the thread's values; NaNs are
// none.  Whole block.
constexpr int kNoCut = 0x7fffffff;
template <int T, class Each>
__device__ __forceinline__ int find_cut(BinScratch<T>& B, int k, int want, Each each, Cut* cut) {
  float lo = __builtin_inff(), hi = -__builtin_inff();
  each([&](float v) {
    if (__builtin_isfinite(v)) {  // (infinities fall into the outer bins)
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
  });
  int count = kNoCut;
#pragma unroll 1
  for (int level = 0; level < 4; ++level) {
    Bins bins;
    if (!make_bins(B, lo, hi, &bins)) break;  // (uniform)
    const float floor = level > 0 ? bins.lo : -__builtin_inff();
    each([&](float v) {
      if (v >= floor) atomicAdd(&B.hist[bins.of(v)], 1);
    });
    __syncthreads();
    int above = 0;
    const int bin = cut_bin(B, k, &above);
    if (bin < 0) break;
    *cut = Cut{bins, floor, bin};
    count = above;
    if (above <= want) break;
    lo = __builtin_inff();
    hi = -__builtin_inff();
    each([&](float v) {
      if (v >= floor && __builtin_isfinite(v) && bins.of(v) == bin) {
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
      }
    });
  }
  __syncthreads();  // (the next make_bins writes what a slow wave may still read in the last)
  return count;
}

// Descending bitonic sort of N = T * E keys, key i = tid * E + e in v[e] of
// thread tid.  Strides below E stay in the thread, those below 64 E in the wave
// (shuffles), the rest (10 stages of 66 at T = 1024, E = 2) cross waves through `lds`
// (N keys).  Whole block.
template <int T, int E>
__device__ __forceinline__ void block_bitonic_desc(uint64_t (&v)[E], uint64_t* lds) {
  const int tid = threadIdx.x;
#pragma unroll 1
  for (int size = 2; size <= T * E; size <<= 1) {
#pragma unroll 1
    for (int stride = size >> 1; stride >= E; stride >>= 1) {
      const int ls = stride / E;  // partner thread: tid ^ ls
      uint64_t o[E];
      if (ls >= kWave) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) lds[e * T + tid] = v[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = lds[e * T + (tid ^ ls)];
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = __shfl_xor(v[e], ls);
      }
      // the lower index keeps the larger key of a pair in a descending run
      const bool lower = (tid & ls) == 0, desc = ((tid * E) & size) == 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const bool big = v[e] > o[e];
        v[e] = (big == (lower == desc)) ? v[e] : o[e];
      }
    }
#pragma unroll
    for (int s = E / 2; s >= 1; s >>= 1) {
      if (s < size) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if ((e & s) == 0) {
            const bool desc = ((tid * E + e) & size) == 0;
            const uint64_t x = v[e], y = v[e | s];
            const bool swap = desc ? x < y : x > y;
            v[e] = swap ? y : x;
            v[e | s] = swap ? x : y;
          }
        }
      }
    }
  }
}

// Sorts the m <= T * E keys get(i) and calls put(i, key) for the first
// min(k, m) of them in descending order.  Whole block; `lds` holds T * E keys
// and may be what get() reads.
template <int T, int E, class Get, class Put>
__device__ __forceinline__ void sort_and_put(int m, int k, uint64_t* lds, Get get, Put put) {
  const int tid = threadIdx.x;
  uint64_t v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = e * T + tid;
    v[e] = i < m ? get(i) : 0ull;  // key 0: below every real key
  }
  __syncthreads();
  block_bitonic_desc<T, E>(v, lds);
  __syncthreads();  // put() may write to lds
  const int top = min(k, m);
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (tid * E + e < top) put(tid * E + e, v[e]);
}

// The same for m <= 256 keys by rank: G threads count the keys above each (over
// slices), two barriers where the network takes 55 stages (rows of 3000 scores,
// k = 10, with their GEMV: 16 -> 8 us).  Equal keys (0: none) rank by position.
template <int T, class Get, class Put>
__device__ __forceinline__ void rank_and_put(int m, int k, uint64_t* lds, Get get, Put put) {
  __shared__ int rank[256];
  const int tid = threadIdx.x;
  const int P = m <= 64 ? 64 : 256, G = T / P;
  const int i = tid & (P - 1), g = tid / P;
  const uint64_t mine = i < m ? get(i) : 0ull;
  if (tid < P) rank[tid] = 0;
  __syncthreads();  // (get() may read from lds)
  if (g == 0 && i < m) lds[i] = mine;
  __syncthreads();
  const int per = (m + G - 1) / G, j1 = min(m, (g + 1) * per);
  int r = 0;
  if (i < m)
#pragma unroll 4
    for (int j = g * per; j < j1; ++j) {
      const uint64_t o = lds[j];
      r += o > mine || (o == mine && j < i) ? 1 : 0;
    }
  if (r > 0) atomicAdd(&rank[i], r);
  __syncthreads();
  if (g == 0 && i < m && rank[i] < k) put(rank[i], mine);
}

template <int T, class Get, class Put>
__device__ __forceinline__ void sort_any(int m, int k, uint64_t* lds, Get get, Put put) {
  if (m <= 256)
    rank_and_put<T>(m, k, lds, get, put);
  else if (m <= T)
    sort_and_put<T, 1>(m, k, lds, get, put);
  else if (m <= 2 * T)
    sort_and_put<T, 2>(m, k, lds, get, put);
  else if (m <= 4 * T)
    sort_and_put<T, 4>(m, k, lds, get, put);
  else
    sort_and_put<T, 8>(m, k, lds, get, put);
}

// The order key of a row's sampled threshold; ~0u: no guess (equal or no finite
// samples).  Whole block.
template <int T>
__device__ __forceinline__ uint32_t sample_threshold(BinScratch<T>& B, const RowTopkArgs& a, const float* src) {
  const int tid = threadIdx.x;
  const int64_t S = 32 * (int64_t)a.groups;  // group g: 32 scores centred in the row's g-th of `groups` parts
  const int64_t step = a.n / a.groups;
  auto at = [&](int64_t i) { return src[(i >> 5) * step + ((step - 32) >> 1) + (i & 31)]; };
  float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll 8
  for (int64_t i = tid; i < S; i += T) {
    const float v = at(i);
    if (__builtin_isfinite(v)) {
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
  }
  Bins bins;
  const bool ok = make_bins(B, lo, hi, &bins);
#pragma unroll 8
  for (int64_t i = tid; i < S; i += T) atomicAdd(&B.hist[bins.of(at(i))], 1);  // (re-read: in cache)
  __syncthreads();
  int above;
  const int b = cut_bin(B, a.rank, &above);
  return ok ? float_order(bins.lo + (float)b / bins.scale) : ~0u;
}

__global__ __launch_bounds__(1024) void row_sample_kernel(RowTopkArgs a) {
  __shared__ BinScratch<1024> B;
  const int r = blockIdx.x;
  const uint32_t tau = sample_threshold(B, a, a.scores + (a.row0 + r) * a.n);
  if (threadIdx.x == 0) {
    a.tau[r] = tau;  // (~0u: no candidates; step 3 streams the row)
    a.count[r] = 0;
  }
}

// Appends the keys of the columns [c0, c1) whose order keys reach tk, kFilterU of
// each of T threads from `base` on: 16-byte loads from the aligned addresses at
// or below each four columns (a row's first column sits `off` floats past one; base =
// c0 - off + a multiple of kFilterU T).  A quad that is not wholly inside the
// range loads its columns one by one.
template <int T, class Put>
__device__ __forceinline__ void filter_round(const float* row, int64_t base, int64_t c0, int64_t c1, uint32_t tk,
                                             int* nbuf, Put put) {
  const int tid = threadIdx.x;
  f32x4 v[kFilterU / 4];
#pragma unroll
  for (int u = 0; u < kFilterU / 4; ++u) {
    const int64_t col = base + (u * T + tid) * 4;
    v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (col >= c0 && col + 4 <= c1) {
      v[u] = *(const f32x4*)(row + col);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (col + j >= c0 && col + j < c1) v[u][j] = row[col + j];
    }
  }
#pragma unroll
  for (int u = 0; u < kFilterU / 4; ++u) {
    const int64_t col = base + (u * T + tid) * 4;
    unsigned pass = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      pass |= (col + j >= c0 && col + j < c1 && float_order(v[u][j]) >= tk ? 1u : 0u) << j;
    if (__ballot(pass != 0) == 0) continue;
    if (pass) {
      int p = atomicAdd(nbuf, __popc(pass));
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((pass >> j) & 1u) put(p++, make_key(v[u][j], (int)(col + j)));
    }
  }
}

__global__ __launch_bounds__(kBlock) void row_filter_kernel(RowTopkArgs a) {
  __shared__ uint64_t buf[kFilterFlush + kFilterRound];
  __shared__ int nbuf, gpos;
  const int tid = threadIdx.x;
  const int r = blockIdx.x / a.chunks;
  const int c = blockIdx.x % a.chunks;
  const int64_t c0 = (int64_t)c * a.len;
  const int64_t c1 = min<int64_t>(c0 + a.len, a.n);
  const float* row = a.scores + (a.row0 + r) * a.n;
  const int off = (int)((reinterpret_cast<uintptr_t>(row) >> 2) & 3);  // (c0: a multiple of 4)
  const uint32_t tk = a.tau[r];
  if (tid == 0) nbuf = 0;
  __syncthreads();
  auto flush = [&]() {  // whole block
    __syncthreads();
    const int m = nbuf;
    if (tid == 0) gpos = atomicAdd(&a.count[r], m);
    __syncthreads();
    const int g = gpos;
    for (int i = tid; i < m; i += kBlock)
      if (g + i < kRowCap) a.cand[(int64_t)r * kRowCap + g + i] = buf[i];
    __syncthreads();
    if (tid == 0) nbuf = 0;
    __syncthreads();
  };
  for (int64_t base = c0 - off; base < c1; base += kFilterRound) {
    filter_round<kBlock>(row, base, c0, c1, tk, &nbuf, [&](int p, uint64_t key) { buf[p] = key; });
    __syncthreads();
    const bool full = nbuf > kFilterFlush;
    if (full) flush();
    else __syncthreads();
  }
  if (nbuf > 0) flush();
}

// kCandidates: the filter's; kShortRow: the row's n <= 8 T scores; either in 64
// registers a thread, so that two rows of 1024 threads share a CU.  Past kNarrowRows rows
// T is the smallest that holds the row: 2500 x 1326, k = 300 79 -> 28 us (T = 1024, 256),
// 2500 x 2600 83 -> 40 (512); 512 rows 1.15 to 0.57 of T = 1024's time, 256 1.4 to 0.7.
// kMidRow: its n <= 2 kRowCap scores, likewise (2386 rows of 10020, k = 2 76 -> 46 us);
// kRow: its n <= kRowDirect scores; kStream: all three steps by the row's one workgroup.
enum Source { kCandidates, kShortRow, kMidRow, kRow, kStream };
template <Source SRC, int T = 1024>
__global__ __launch_bounds__(T, SRC == kRow ? 1 : 8) void row_final_kernel(RowTopkArgs a) {
  constexpr bool DIRECT = SRC != kCandidates && SRC != kStream;
  constexpr int E = 8, kCap = T * E;
  __shared__ uint64_t keys[kCap];
  __shared__ BinScratch<T> B;
  __shared__ int nbuf;
  __shared__ uint64_t kth;
  const int tid = threadIdx.x;
  const int r = blockIdx.x;
  const int k = a.k;
  const float* row = a.scores + (a.row0 + r) * a.n;
  const int64_t obase = (a.row0 + r) * (int64_t)k;
  auto put = [&](int i, uint64_t key) {
    const bool none = key == 0ull;  // (a skipped NaN)
    a.out_v[obase + i] = none ? -__builtin_inff() : key_score(key);
    const int id = none ? -1 : key_id(key);
    if (a.ids64)
      ((int64_t*)a.out_i)[obase + i] = id;
    else
      ((int*)a.out_i)[obase + i] = id;
  };
  // A NaN that counts stands beyond the infinity of its sign in the keys' order: f() gets that.
  auto ordered = [&](float v) { return v == v || a.skip_nan ? v : __builtin_copysignf(__builtin_inff(), v); };
  // Writes the k best of the values in the threads' registers: each(f) calls
  // f(value, e) for the thread's own, key(e) is its key.  A sort of thousands of
  // keys costs several times one of the ~k that matter, so they are cut first: to
  // those that reach the k-th best of the threads' maxima (one value a thread to
  // bin), or, where that leaves too many or k is large, by bins of their own.
  // False when neither leaves kCap, unless `all` fit.  (Searches over 16000 x
  // 768, 200 queries, k = 10, plain / one row of 3000 times the others' norm: 27 / 29 us;
  // with bins over the row's values alone 32 / 144.)
  auto finish = [&](auto each, auto key, bool all) __attribute__((always_inline)) {
    Cut cut;
    int total = kNoCut;
    if (k <= T / 2) {
      float mx = -__builtin_inff();
      bool any = false;
      each([&](float v, int) {
        any = true;
        mx = fmaxf(mx, v);
      });
      const int c = find_cut(B, k, 2 * k + 32, [&](auto f) {
        if (any) f(mx);
      }, &cut);
      if (c != kNoCut) {  // (uniform)
        float t = wave_min_f32(any && cut.keeps(mx) ? mx : __builtin_inff());
        if (tid % kWave == 0) B.mm[0][tid / kWave] = t;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < T / kWave; ++i) t = fminf(t, B.mm[0][i]);
        each([&](float v, int e) {
          if (v >= t) {
            const int p = atomicAdd(&nbuf, 1);
            if (p < kCap) keys[p] = key(e);
          }
        });
        __syncthreads();
        total = nbuf;
        if (total > kCap) {
          __syncthreads();
          if (tid == 0) nbuf = 0;
          __syncthreads();
        }
      }
    }
    if (total > kCap) {
      const int most = k + k / 8;  // the smallest network that holds these
      const int c = find_cut(B, k, most <= 2 * T ? 2 * T : most <= 4 * T ? 4 * T : kCap, [&](auto f) {
        each([&](float v, int) { f(v); });
      }, &cut);
      if (c > kCap && !all) return false;
      each([&](float v, int e) {
        if (c > kCap || cut.keeps(v)) keys[atomicAdd(&nbuf, 1)] = key(e);
      });
      __syncthreads();
      total = nbuf;
    }
    if constexpr (SRC == kMidRow || SRC == kRow)
      if (!a.skip_nan) {  // (an infinity may have been a NaN)
#pragma unroll 1
        for (int i = tid; i < total; i += T)
          if (!__builtin_isfinite(key_score(keys[i]))) keys[i] = make_key(row[key_id(keys[i])], key_id(keys[i]));
        __syncthreads();
      }
    sort_any<T>(total, k, keys, [&](int i) { return keys[i]; }, put);
    for (int i = total + tid; i < k; i += T) put(i, 0ull);  // (NaNs left out)
    return true;
  };
  if (tid == 0) nbuf = 0;
  int m = (int)a.n;
  if constexpr (SRC == kCandidates) m = a.count[r];
  if constexpr (SRC == kStream) {
    const uint32_t tk = sample_threshold(B, a, row);  // (its barriers: nbuf is cleared)
    const int off = (int)((reinterpret_cast<uintptr_t>(row) >> 2) & 3);
    if (tk != ~0u)
      for (int64_t base = -off; base < a.n; base += T * kFilterU) {
        filter_round<T>(row, base, 0, a.n, tk, &nbuf, [&](int p, uint64_t key) {
          if (p < kCap) keys[p] = key;
        });
        if (*(volatile int*)&nbuf > kCap) break;
      }
    __syncthreads();
    m = nbuf;
    __syncthreads();
    if (tid == 0) nbuf = 0;
  }
  if constexpr (SRC == kMidRow || SRC == kRow) {
    constexpr int R = (SRC == kMidRow ? 2 * kRowCap : kRowDirect) / T;
    float v[R];
#pragma unroll
    for (int e = 0; e < R; ++e) v[e] = e * T < m ? row[min(e * T + tid, m - 1)] : 0.f;
#pragma unroll
    for (int e = 0; e < R; ++e) v[e] = ordered(v[e]);  // (after all loads: with them 8.5 -> 11.8 us, 200 rows of 16000)
    auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < R; ++e)
        if (e * T + tid < m) f(v[e], e);
    };
    if (finish(each, [&](int e) { return make_key(v[e], e * T + tid); }, false)) return;
    __syncthreads();
  } else if (DIRECT || (m >= k && m <= kCap)) {
    const uint64_t* cand = SRC == kStream ? keys : DIRECT ? nullptr : a.cand + (int64_t)r * kRowCap;
    auto get = [&](int i) -> uint64_t {
      if constexpr (!DIRECT) return cand[i];
      const float v = row[i];
      return a.skip_nan && v != v ? 0ull : make_key(v, i);
    };
    if (m <= 256 || (m <= 2 * T && (4 * k > m || T == kNarrow))) {
      sort_any<T>(m, k, keys, get, put);
      return;
    }
    uint64_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = e * T + tid;
      v[e] = i < m ? get(i) : 0ull;
    }
    if constexpr (SRC == kStream) __syncthreads();  // (read before finish() writes to keys)
    auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (e * T + tid < m) f(ordered(key_score(v[e])), e);
    };
    finish(each, [&](int e) { return v[e]; }, true);
    return;
  }
  // The threshold missed, or the cut (equal scores, NaNs): the row streamed, its running k best in LDS.
  if (tid == 0) kth = 0ull;
  __syncthreads();
  constexpr int kSkip = 32768;  // columns left out at once when none reaches the running k best
  int64_t probe = 0;            // the next column from which that is tried
  for (int64_t base = 0; base < a.n; base += 4 * T) {
    const uint64_t t = kth;
    auto key_of = [&](float v, int64_t col) { return a.skip_nan && v != v ? 0ull : make_key(v, (int)col); };
    if (t != 0ull && base >= probe && base + kSkip < a.n) {  // (uniform)
      bool any = false;
#pragma unroll 1
      for (int i = 0; i < kSkip; i += 16 * T) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = row[base + i + u * T + tid];
#pragma unroll
        for (int u = 0; u < 16; ++u) any |= key_of(v[u], base + i + u * T + tid) > t;
      }
      if (!__syncthreads_or(any)) {
        base += kSkip - 4 * T;
        continue;
      }
      probe = base + kSkip;
    }
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t col = base + u * T + tid;
      v[u] = row[col < a.n ? col : a.n - 1];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t col = base + u * T + tid;
      const uint64_t key = col < a.n ? key_of(v[u], col) : 0ull;
      if (key > t) keys[atomicAdd(&nbuf, 1)] = key;
    }
    __syncthreads();
    const int nb = nbuf;
    const bool last = base + 4 * T >= a.n;
    if (last) {
      sort_any<T>(nb, k, keys, [&](int i) { return keys[i]; }, put);
      for (int i = nb + tid; i < k; i += T) put(i, 0ull);  // (NaNs left out)
    } else if (nb > 4 * T) {
      sort_and_put<T, E>(nb, k, keys, [&](int i) { return keys[i]; }, [&](int i, uint64_t key) {
        keys[i] = key;
        if (i == k - 1) kth = key;
      });
      if (tid == 0) nbuf = k;
    }
    __syncthreads();
  }
}

}  // namespace

hipError_t launch_row_topk(const RowTopkArgs& a, int rows, hipStream_t s) {
  if (a.k < 1 || a.k > kRowTopkMaxK || a.n < a.k || rows < 1 || a.scores == nullptr) return hipErrorInvalidValue;
  const bool sampled = a.n > kRowDirect;
  if (sampled && (a.groups < 1 || 32 * (int64_t)a.groups > a.n)) return hipErrorInvalidValue;
  if (!sampled || a.narrow) {
    constexpr int64_t kMost = 1 << 21;  // workgroups of a launch: fewer than 2^32 threads
    for (int64_t r = 0; r < rows; r += kMost) {
      RowTopkArgs b = a;
      b.row0 = a.row0 + r;
      const dim3 grid((unsigned)(rows - r < kMost ? rows - r : kMost));
      if (sampled)
        hipLaunchKernelGGL((row_final_kernel<kStream, kNarrow>), grid, dim3(kNarrow), 0, s, b);
      else if (a.n <= 8 * kNarrow && rows > kNarrowRows)
        hipLaunchKernelGGL((row_final_kernel<kShortRow, kNarrow>), grid, dim3(kNarrow), 0, s, b);
      else if (a.n <= 8 * 512 && rows > kNarrowRows)
        hipLaunchKernelGGL((row_final_kernel<kShortRow, 512>), grid, dim3(512), 0, s, b);
      else if (a.n <= kRowCap)
        hipLaunchKernelGGL(row_final_kernel<kShortRow>, grid, dim3(1024), 0, s, b);
      else if (a.n <= 2 * kRowCap)
        hipLaunchKernelGGL(row_final_kernel<kMidRow>, grid, dim3(1024), 0, s, b);
      else
        hipLaunchKernelGGL(row_final_kernel<kRow>, grid, dim3(1024), 0, s, b);
      if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  if (a.tau == nullptr || a.count == nullptr || a.cand == nullptr || a.chunks < 1 || a.len < 1 ||
      a.len * a.chunks < a.n || (int64_t)rows * a.chunks > 0x7fffffff)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(row_sample_kernel, dim3(rows), dim3(1024), 0, s, a);
  hipLaunchKernelGGL(row_filter_kernel, dim3(rows * a.chunks), dim3(kBlock), 0, s, a);
  hipLaunchKernelGGL(row_final_kernel<kCandidates>, dim3(rows), dim3(1024), 0, s, a);
  return hipGetLastError();
}

}  // namespace cvs
