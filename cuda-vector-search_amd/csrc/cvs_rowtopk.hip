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
//
// Measured against chunk-wise radix selects and a merge of the chunks' top k:
// 64 rows x 300k, k = 1000: 189 -> 49 us; 1 x 4M, k = 1000: 3380 -> 60 us; whole
// rows, 1000 x 8000, k = 1000: 77 -> 45 us.
#include "cvs_common.h"
#include "cvs_kernels.h"

namespace cvs {

namespace {

constexpr int kFinal = 1024;              // threads of the sample and final kernels
constexpr int kFinalWaves = kFinal / kWave;
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

struct BinScratch {
  float mm[2][kFinalWaves];
  int hist[kBins];
  int wsum[kFinalWaves];
  int bin, above;
};

// The block's bins over the [min, max] of every thread's (lo, hi), an empty
// histogram, and false when that range is empty or not finite.  Whole block.
__device__ __forceinline__ bool make_bins(BinScratch& B, float lo, float hi, Bins* bins) {
  const int tid = threadIdx.x;
  lo = wave_min_f32(lo);
  hi = wave_max_f32(hi);
  if (tid % kWave == 0) {
    B.mm[0][tid / kWave] = lo;
    B.mm[1][tid / kWave] = hi;
  }
  B.hist[tid] = 0;  // kBins == kFinal
  __syncthreads();
  lo = B.mm[0][0];
  hi = B.mm[1][0];
#pragma unroll
  for (int i = 1; i < kFinalWaves; ++i) {
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
__device__ __forceinline__ int cut_bin(BinScratch& B, int want, int* above) {
  const int tid = threadIdx.x;
  const int b = kBins - 1 - tid;  // descending
  const int c = B.hist[b];
  int incl = wave_incl_sum_i32(c);
  if (tid % kWave == kWave - 1) B.wsum[tid / kWave] = incl;
  if (tid == 0) B.bin = -1;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kFinalWaves; ++w) incl += w < tid / kWave ? B.wsum[w] : 0;
  if (incl - c < want && want <= incl) {
    B.bin = b;
    B.above = incl;
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
// values, all equal, NaNs that count).  each(f) calls f(v) for the thread's
// values.  Whole block.
constexpr int kNoCut = 0x7fffffff;
template <class Each>
__device__ __forceinline__ int find_cut(BinScratch& B, int k, int want, bool skip_nan, Each each, Cut* cut) {
  float lo = __builtin_inff(), hi = -__builtin_inff();
  each([&](float v) {
    if (__builtin_isfinite(v)) {  // (infinities fall into the outer bins)
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    } else if (v != v && !skip_nan) {
      hi = __builtin_inff();  // above +inf in the keys' order: no bin
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

// Descending bitonic sort of N = kFinal * E keys, key i = tid * E + e in v[e] of
// thread tid.  Strides below E stay in the thread, those below 64 E in the wave
// (shuffles), the rest (10 stages of 66 at E = 2) cross waves through `lds`
// (N keys).  Whole block.
template <int E>
__device__ __forceinline__ void block_bitonic_desc(uint64_t (&v)[E], uint64_t* lds) {
  const int tid = threadIdx.x;
#pragma unroll 1
  for (int size = 2; size <= kFinal * E; size <<= 1) {
#pragma unroll 1
    for (int stride = size >> 1; stride >= E; stride >>= 1) {
      const int ls = stride / E;  // partner thread: tid ^ ls
      uint64_t o[E];
      if (ls >= kWave) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) lds[e * kFinal + tid] = v[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = lds[e * kFinal + (tid ^ ls)];
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

// Sorts the m <= kFinal * E keys get(i) and calls put(i, key) for the first
// min(k, m) of them in descending order.  Whole block; `lds` holds kFinal * E keys
// and may be what get() reads.
template <int E, class Get, class Put>
__device__ __forceinline__ void sort_and_put(int m, int k, uint64_t* lds, Get get, Put put) {
  const int tid = threadIdx.x;
  uint64_t v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = e * kFinal + tid;
    v[e] = i < m ? get(i) : 0ull;  // key 0: below every real key
  }
  __syncthreads();
  block_bitonic_desc<E>(v, lds);
  __syncthreads();  // put() may write to lds
  const int top = min(k, m);
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (tid * E + e < top) put(tid * E + e, v[e]);
}

// The same for m <= 256 keys by rank: G threads count the keys above each (over
// slices), two barriers where the network takes 55 stages (rows of 3000 scores,
// k = 10, with their GEMV: 16 -> 8 us).  Equal keys (0: none) rank by position.
template <class Get, class Put>
__device__ __forceinline__ void rank_and_put(int m, int k, uint64_t* lds, Get get, Put put) {
  __shared__ int rank[256];
  const int tid = threadIdx.x;
  const int P = m <= 64 ? 64 : 256, G = kFinal / P;
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

template <class Get, class Put>
__device__ __forceinline__ void sort_any(int m, int k, uint64_t* lds, Get get, Put put) {
  if (m <= 256)
    rank_and_put(m, k, lds, get, put);
  else if (m <= kFinal)
    sort_and_put<1>(m, k, lds, get, put);
  else if (m <= 2 * kFinal)
    sort_and_put<2>(m, k, lds, get, put);
  else if (m <= 4 * kFinal)
    sort_and_put<4>(m, k, lds, get, put);
  else
    sort_and_put<8>(m, k, lds, get, put);
}

__global__ __launch_bounds__(kFinal) void row_sample_kernel(RowTopkArgs a) {
  __shared__ BinScratch B;
  const int tid = threadIdx.x;
  const int r = blockIdx.x;
  const float* src = a.scores + (a.row0 + r) * a.n;
  const int64_t S = 32 * (int64_t)a.groups;  // group g: 32 scores centred in the row's g-th of `groups` parts
  const int64_t step = a.n / a.groups;
  auto at = [&](int64_t i) { return src[(i >> 5) * step + ((step - 32) >> 1) + (i & 31)]; };
  float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll 8
  for (int64_t i = tid; i < S; i += kFinal) {
    const float v = at(i);
    if (__builtin_isfinite(v)) {
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
  }
  Bins bins;
  const bool ok = make_bins(B, lo, hi, &bins);
#pragma unroll 8
  for (int64_t i = tid; i < S; i += kFinal) atomicAdd(&B.hist[bins.of(at(i))], 1);  // (re-read: in cache)
  __syncthreads();
  int above;
  const int b = cut_bin(B, a.rank, &above);
  if (tid == 0) {
    // (equal or no finite samples: no guess, and no candidates; step 3 streams the row)
    a.tau[r] = ok ? float_order(bins.lo + (float)b / bins.scale) : ~0u;
    a.count[r] = 0;
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
  // 16-byte loads from the aligned addresses at or below each four columns: a
  // row's first column sits `off` floats past one.  A quad that is not wholly
  // inside the chunk loads its columns one by one.
  const int off = (int)((reinterpret_cast<uintptr_t>(row) >> 2) & 3);
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
    f32x4 v[kFilterU / 4];
#pragma unroll
    for (int u = 0; u < kFilterU / 4; ++u) {
      const int64_t col = base + (u * kBlock + tid) * 4;
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
      const int64_t col = base + (u * kBlock + tid) * 4;
      unsigned pass = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        pass |= (col + j >= c0 && col + j < c1 && float_order(v[u][j]) >= tk ? 1u : 0u) << j;
      if (__ballot(pass != 0) == 0) continue;
      if (pass) {
        int p = atomicAdd(&nbuf, __popc(pass));
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if ((pass >> j) & 1u) buf[p++] = make_key(v[u][j], (int)(col + j));
      }
    }
    __syncthreads();
    const bool full = nbuf > kFilterFlush;
    if (full) flush();
    else __syncthreads();
  }
  if (nbuf > 0) flush();
}

// kCandidates: the filter's; kShortRow: the row's n <= kRowCap scores; either in 64
// registers a thread, so that two rows share a CU (1130 rows of 1721, k = 278 63 -> 43 us);
// kMidRow: its n <= 2 kRowCap scores, likewise (2386 rows of 10020, k = 2 76 -> 46 us);
// kRow: its n <= kRowDirect scores.
enum Source { kCandidates, kShortRow, kMidRow, kRow };
template <Source SRC>
__global__ __launch_bounds__(kFinal, SRC == kRow ? 1 : 8) void row_final_kernel(RowTopkArgs a) {
  constexpr bool DIRECT = SRC != kCandidates;
  constexpr int E = kRowCap / kFinal;
  __shared__ uint64_t keys[kRowCap];
  __shared__ BinScratch B;
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
  // Writes the k best of the values in the threads' registers: each(f) calls
  // f(value, e) for the thread's own, key(e) is its key.  A sort of thousands of
  // keys costs several times one of the ~k that matter, so they are cut first: to
  // those that reach the k-th best of the threads' maxima (one value a thread to
  // bin), or, where that leaves too many or k is large, by bins of their own.
  // False when neither leaves kRowCap, unless `all` fit.  (Searches over 16000 x
  // 768, 200 queries, k = 10, plain / one row of 3000 times the others' norm: 27 / 29 us;
  // with bins over the row's values alone 32 / 144.)
  auto finish = [&](auto each, auto key, bool all) __attribute__((always_inline)) {
    Cut cut;
    int total = kNoCut;
    if (k <= kFinal / 2) {
      float mx = -__builtin_inff();
      bool any = false, nan = false;
      each([&](float v, int) {
        any = true;
        nan |= v != v;
        mx = fmaxf(mx, v);
      });
      if (nan && !a.skip_nan) mx = __builtin_nanf("");
      const int c = find_cut(B, k, 2 * k + 32, a.skip_nan, [&](auto f) {
        if (any) f(mx);
      }, &cut);
      if (c != kNoCut) {  // (uniform)
        float t = wave_min_f32(any && cut.keeps(mx) ? mx : __builtin_inff());
        if (tid % kWave == 0) B.mm[0][tid / kWave] = t;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kFinalWaves; ++i) t = fminf(t, B.mm[0][i]);
        each([&](float v, int e) {
          if (v >= t) {
            const int p = atomicAdd(&nbuf, 1);
            if (p < kRowCap) keys[p] = key(e);
          }
        });
        __syncthreads();
        total = nbuf;
        if (total > kRowCap) {
          __syncthreads();
          if (tid == 0) nbuf = 0;
          __syncthreads();
        }
      }
    }
    if (total > kRowCap) {
      const int c = find_cut(B, k, 2 * kFinal, a.skip_nan, [&](auto f) {
        each([&](float v, int) { f(v); });
      }, &cut);
      if (c > kRowCap && !all) return false;
      each([&](float v, int e) {
        if (c > kRowCap || cut.keeps(v)) keys[atomicAdd(&nbuf, 1)] = key(e);
      });
      __syncthreads();
      total = nbuf;
    }
    sort_any(total, k, keys, [&](int i) { return keys[i]; }, put);
    for (int i = total + tid; i < k; i += kFinal) put(i, 0ull);  // (NaNs left out)
    return true;
  };
  const int m = DIRECT ? (int)a.n : a.count[r];
  if (tid == 0) nbuf = 0;
  if constexpr (SRC == kMidRow || SRC == kRow) {
    constexpr int R = (SRC == kMidRow ? 2 * kRowCap : kRowDirect) / kFinal;
    float v[R];
#pragma unroll
    for (int e = 0; e < R; ++e) v[e] = e * kFinal < m ? row[min(e * kFinal + tid, m - 1)] : 0.f;
    auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < R; ++e)
        if (e * kFinal + tid < m) f(v[e], e);
    };
    if (finish(each, [&](int e) { return make_key(v[e], e * kFinal + tid); }, false)) return;
    __syncthreads();
  } else if (DIRECT || (m >= k && m <= kRowCap)) {
    const uint64_t* cand = DIRECT ? nullptr : a.cand + (int64_t)r * kRowCap;
    auto get = [&](int i) -> uint64_t {
      if constexpr (!DIRECT) return cand[i];
      const float v = row[i];
      return a.skip_nan && v != v ? 0ull : make_key(v, i);
    };
    if (m <= 256 || (m <= 2 * kFinal && 4 * k > m)) {
      sort_any(m, k, keys, get, put);
      return;
    }
    uint64_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = e * kFinal + tid;
      v[e] = i < m ? get(i) : 0ull;
    }
    auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (e * kFinal + tid < m) f(key_score(v[e]), e);
    };
    finish(each, [&](int e) { return v[e]; }, true);
    return;
  }
  // The threshold missed, or the cut (equal scores, NaNs): the row streamed, its running k best in LDS.
  if (tid == 0) kth = 0ull;
  __syncthreads();
  constexpr int kSkip = 16 * kFinal;  // columns left out at once when none reaches the running k best
  for (int64_t base = 0; base < a.n; base += 4 * kFinal) {
    const uint64_t t = kth;
    auto key_at = [&](int64_t col) -> uint64_t {
      const float v = col < a.n ? row[col] : 0.f;
      return col < a.n && !(a.skip_nan && v != v) ? make_key(v, (int)col) : 0ull;
    };
    if (t != 0ull && base % kSkip == 0 && base + kSkip < a.n) {  // (uniform)
      bool any = false;
#pragma unroll
      for (int u = 0; u < kSkip / kFinal; ++u) any |= key_at(base + u * kFinal + tid) > t;
      if (!__syncthreads_or(any)) {
        base += kSkip - 4 * kFinal;
        continue;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint64_t key = key_at(base + u * kFinal + tid);
      if (key > t) keys[atomicAdd(&nbuf, 1)] = key;
    }
    __syncthreads();
    const int nb = nbuf;
    const bool last = base + 4 * kFinal >= a.n;
    if (last) {
      sort_any(nb, k, keys, [&](int i) { return keys[i]; }, put);
      for (int i = nb + tid; i < k; i += kFinal) put(i, 0ull);  // (NaNs left out)
    } else if (nb > 4 * kFinal) {
      sort_and_put<E>(nb, k, keys, [&](int i) { return keys[i]; }, [&](int i, uint64_t key) {
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
  if (a.n <= kRowDirect) {
    constexpr int64_t kMost = 1 << 21;  // workgroups of a launch: fewer than 2^32 threads
    for (int64_t r = 0; r < rows; r += kMost) {
      RowTopkArgs b = a;
      b.row0 = a.row0 + r;
      const dim3 grid((unsigned)(rows - r < kMost ? rows - r : kMost));
      if (a.n <= kRowCap)
        hipLaunchKernelGGL(row_final_kernel<kShortRow>, grid, dim3(kFinal), 0, s, b);
      else if (a.n <= 2 * kRowCap)
        hipLaunchKernelGGL(row_final_kernel<kMidRow>, grid, dim3(kFinal), 0, s, b);
      else
        hipLaunchKernelGGL(row_final_kernel<kRow>, grid, dim3(kFinal), 0, s, b);
      if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  if (a.tau == nullptr || a.count == nullptr || a.cand == nullptr || a.groups < 1 || 32 * (int64_t)a.groups > a.n ||
      a.chunks < 1 || a.len < 1 || a.len * a.chunks < a.n || (int64_t)rows * a.chunks > 0x7fffffff)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(row_sample_kernel, dim3(rows), dim3(kFinal), 0, s, a);
  hipLaunchKernelGGL(row_filter_kernel, dim3(rows * a.chunks), dim3(kBlock), 0, s, a);
  hipLaunchKernelGGL(row_final_kernel<kCandidates>, dim3(rows), dim3(kFinal), 0, s, a);
  return hipGetLastError();
}

}  // namespace cvs
