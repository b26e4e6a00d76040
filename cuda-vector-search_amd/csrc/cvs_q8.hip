// int8 companion of the fp16 corpus and of each query batch, for the int8
// pre-filter of the exact search (no counterpart in the reference, whose only
// corpus format is the fp16 matrix of cuda_vector_search/index.py:56-78).
//
// Rows are quantised symmetrically: a 64-row block of the corpus shares one
// scale s_b = max|x| / 127 over the block, a query row has its own s_q, and
// x~ = rint(x * (127 / max)) in [-127, 127].  The scan then computes
// A = s_q * s_b * sum(q~ x~) with int8 MFMAs (exact int32 sums), and
//
//     |q.x - A| <= |q^|_2 |f|_2 + |e|_2 |x|_2,   q^ = s_q q~, e = q - q^,
//                                                 f = x - s_b x~
//
// (Cauchy-Schwarz on the two residuals), so the exact score of every row lies
// within that slack of A.  The kernels here store, per block, s_b and upper
// bounds of max |f_r|_2 and max |x_r|_2 over its rows, and per query s_q,
// |q^|_2 and |e|_2 (norms rounded up to cover fp32 accumulation).
//
// The companion holds the rows in ascending order of their largest magnitude
// max_j |x_rj| (a stable sort: equal maxima keep the corpus order), so that
// the rows sharing a block, and its scale s_b, have nearly the same maximum:
// |f_r| then tracks each row's own scale instead of the largest of 64 random
// rows (for unit rows of width 768, max |f_r| per block drops by ~23% and the
// slack by ~13%).  perm[r] is the corpus row at companion row r.
#include <rocprim/device/device_radix_sort.hpp>

#include "cvs_common.h"
#include "cvs_kernels.h"
#include "cvs_q8_row.h"

namespace cvs {

namespace {

constexpr float kNormUp = 1.0f + 1.0f / 2048.0f;  // > 1 + d * 2^-24 for d <= 8192, plus sqrt's ulp


// Sort keys: the fp16 bit pattern of max_j |x_rj| (non-negative halves order
// like their bit patterns; NaNs are skipped as fmaxf skips them), 16 lanes per
// row, and the row ids to carry along.
__global__ __launch_bounds__(kBlock) void q8_rowkey_kernel(const _Float16* x, int64_t n, int d, uint16_t* key,
                                                           int* ids, float* xmax) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *xmax = 0.f;  // (q8_build_kernel takes the maximum into it)
  const int64_t row = (int64_t)blockIdx.x * (kBlock / 16) + (threadIdx.x >> 4);
  const int l16 = threadIdx.x & 15;
  float m = 0.f;
  if (row < n) {
    const half8* src = reinterpret_cast<const half8*>(x + row * (int64_t)d);
    for (int p = l16; p < d / 8; p += 16) {
      const half8 v = src[p];
#pragma unroll
      for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf((float)v[j]));
    }
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (row < n && l16 == 0) {
    key[row] = __builtin_bit_cast(uint16_t, (_Float16)m);  // m is a half's magnitude: exact
    ids[row] = (int)row;
  }
}

// The largest magnitude of each 64-row block, the last of its rows in the sort's
// ascending keys, into bmeta[blk].w (key is overwritten by the int8 rows), and
// perm[r] = r for the padding rows r in [n, rows).
__global__ __launch_bounds__(kBlock) void q8_block_max_kernel(const uint16_t* key, int* perm, float4* bmeta, int64_t n,
                                                              int64_t nblk) {
  const int64_t blk = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (blk >= nblk) return;
  const int64_t last = min(64 * blk + 64, n) - 1;
  bmeta[blk].w = (float)__builtin_bit_cast(_Float16, key[last]);
  if (blk == nblk - 1)
    for (int64_t r = n; r < 64 * nblk; ++r) perm[r] = (int)r;
}

// One workgroup per 64-row block of the companion, 8 lanes per row, which read
// corpus row perm[r] once, 128 bytes per load and kQ8Loads loads in flight, with
// the block's scale known beforehand (q8_block_max_kernel), write the int8 row
// and its zero padding and sum the row's norms.  Memory-bound: 2 d bytes read
// and dq written per row.  Holding a block's rows in registers for both passes
// (the scale found here) left one workgroup per CU at d = 1024: 1140 us for
// 300k rows.  The whole companion build (row keys, sort, blocks), against 4
// lanes a row and rows read twice: 500k x 768 744 -> 431 us, 300k x 1024 670 ->
// 402 us, 500k x 384 369 -> 248 us; narrow rows skip the pieces of padding (296k x
// 128 130 -> 115).
constexpr int kQ8Loads = 6;  // 8-element pieces per lane and round (dq is a multiple of 64 * 6)
__global__ __launch_bounds__(512) void q8_build_kernel(Q8BuildArgs a) {
  constexpr int NW = 512 / kWave;
  __shared__ float fmax_s[NW], xmax_s[NW];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int64_t blk = blockIdx.x;
  const int64_t row = blk * 64 + (tid >> 3);
  const int part = tid & 7;
  const bool live = row < a.n;
  const int np = a.d / 64;  // a lane's pieces
  const half8* src = reinterpret_cast<const half8*>(a.x + (live ? a.perm[row] : 0) * (int64_t)a.d) + part;
  const float M = a.bmeta[blk].w;
  const float s = M / 127.f;
  const float inv = M > 0.f ? 127.f / M : 0.f;

  signed char* dst = a.xq + row * (int64_t)a.dq + 8 * part;
  float ff = 0.f, xx = 0.f;
#pragma unroll 1
  for (int i0 = 0; 64 * i0 < a.dq; i0 += kQ8Loads) {
    half8 v[kQ8Loads];
#pragma unroll
    for (int i = 0; i < kQ8Loads; ++i) v[i] = i0 + i < np ? src[8 * (i0 + i)] : half8{};  // (uniform: they issue together)
#pragma unroll
    for (int i = 0; i < kQ8Loads; ++i) {
      unsigned lo = 0, hi = 0;
      if (i0 + i < np) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float xv = live ? (float)v[i][j] : 0.f;
          const signed char c = q8_quant(xv, inv);
          const float f = fmaf(-s, (float)c, xv);
          ff = fmaf(f, f, ff);
          xx = fmaf(xv, xv, xx);
          if (j < 4) lo |= (unsigned)(unsigned char)c << (8 * j);
          else hi |= (unsigned)(unsigned char)c << (8 * (j - 4));
        }
      }
      *reinterpret_cast<int2*>(dst + 64 * (i0 + i)) = int2{(int)lo, (int)hi};  // (zero past d)
    }
  }
  // row norms: the row's 8 threads are consecutive lanes
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) {
    ff += __shfl_xor(ff, off);
    xx += __shfl_xor(xx, off);
  }
  float fn = sqrtf(ff) * kNormUp, xn = sqrtf(xx) * kNormUp;
#pragma unroll
  for (int off = kWave / 2; off >= 8; off >>= 1) {
    fn = fmaxf(fn, __shfl_xor(fn, off));
    xn = fmaxf(xn, __shfl_xor(xn, off));
  }
  if (lane == 0) {
    fmax_s[w] = fn;
    xmax_s[w] = xn;
  }
  __syncthreads();
  if (tid == 0) {
    float4 meta = float4{s, fmax_s[0], xmax_s[0], 0.f};
#pragma unroll
    for (int i = 1; i < NW; ++i) {
      meta.y = fmaxf(meta.y, fmax_s[i]);
      meta.z = fmaxf(meta.z, xmax_s[i]);
    }
    a.bmeta[blk] = meta;
    // the corpus-wide maximum: non-negative floats order like their bits (a NaN norm is left out)
    // (A look first: thousands of atomics on one word queue up.  A stale value is only a smaller one.)
    if (meta.z > *reinterpret_cast<volatile float*>(a.xmax))
      atomicMax(reinterpret_cast<int*>(a.xmax), __float_as_int(meta.z));
  }
}

// One wave per query row; the whole grid also clears a.zero[0, nzero).
__global__ __launch_bounds__(kBlock) void q8_query_kernel(Q8QueryArgs a) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < a.nzero; i += (int64_t)gridDim.x * kBlock)
    a.zero[i] = 0ull;
  const int64_t r = (int64_t)blockIdx.x * (kBlock / kWave) + (threadIdx.x >> 6);
  if (r >= a.nq) return;  // whole wave
  q8_query_row(a.q + r * a.d, a.d, a.dq, a.qq + r * a.dq, a.qmeta + r, threadIdx.x & 63, a.qf, r);
}

}  // namespace

// Row order, then the blocks.  The sort's key and id buffers and its scratch
// live in the companion's own int8-row region (rows * dq >= 384 n bytes, far
// more than the ~14 n bytes they take), which q8_build_kernel overwrites only
// after the sort, in stream order: the build allocates nothing.
namespace {
struct Q8SortBufs {
  uint16_t *key_in, *key_out;
  int* ids;
  void* tmp;
  size_t sort_bytes;
};
hipError_t q8_sort_bufs(const Q8BuildArgs& a, Q8SortBufs* b, hipStream_t s) {
  if (a.d < 64 || a.d % 64 != 0 || a.d > 1536 || a.dq < a.d || a.dq % (64 * kQ8Loads) != 0 || a.dq > 1536 || a.perm == nullptr)
    return hipErrorInvalidValue;
  if (a.n < 1 || a.n >= 0x7fffffff) return hipErrorInvalidValue;
  b->sort_bytes = 0;
  hipError_t e = rocprim::radix_sort_pairs(nullptr, b->sort_bytes, (const uint16_t*)nullptr, (uint16_t*)nullptr,
                                           (const int*)nullptr, (int*)nullptr, (unsigned)a.n, 0, 15, s);
  if (e != hipSuccess) return e;
  const size_t keys_bytes = ((size_t)a.n * sizeof(uint16_t) + 255) / 256 * 256;
  const size_t ids_bytes = ((size_t)a.n * sizeof(int) + 255) / 256 * 256;
  const size_t rows = ((size_t)a.n + 63) / 64 * 64;
  if (2 * keys_bytes + ids_bytes + b->sort_bytes > rows * (size_t)a.dq) return hipErrorInvalidValue;
  char* buf = reinterpret_cast<char*>(a.xq);
  b->key_in = reinterpret_cast<uint16_t*>(buf);
  b->key_out = reinterpret_cast<uint16_t*>(buf + keys_bytes);
  b->ids = reinterpret_cast<int*>(buf + 2 * keys_bytes);
  b->tmp = buf + 2 * keys_bytes + ids_bytes;
  return hipSuccess;
}
}  // namespace

hipError_t q8_build_keys(const Q8BuildArgs& a, PrepArgs* p, hipStream_t s) {
  Q8SortBufs b;
  hipError_t e = q8_sort_bufs(a, &b, s);
  if (e != hipSuccess) return e;
  p->key = b.key_in;
  p->ids = b.ids;
  p->xmax = a.xmax;
  return hipSuccess;
}

hipError_t launch_q8_build(const Q8BuildArgs& a, bool keyed, hipStream_t s) {
  Q8SortBufs b;
  hipError_t e = q8_sort_bufs(a, &b, s);
  if (e != hipSuccess) return e;
  if (!keyed) {
    const int per = kBlock / 16;
    hipLaunchKernelGGL(q8_rowkey_kernel, dim3((unsigned)((a.n + per - 1) / per)), dim3(kBlock), 0, s, a.x, a.n, a.d,
                       b.key_in, b.ids, a.xmax);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  e = rocprim::radix_sort_pairs(b.tmp, b.sort_bytes, b.key_in, b.key_out, b.ids, a.perm, (unsigned)a.n, 0, 15, s);
  if (e != hipSuccess) return e;
  const int64_t nblk = (a.n + 63) / 64;
  hipLaunchKernelGGL(q8_block_max_kernel, dim3((unsigned)((nblk + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, b.key_out,
                     a.perm, a.bmeta, a.n, nblk);
  hipLaunchKernelGGL(q8_build_kernel, dim3((unsigned)nblk), dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_q8_queries(const Q8QueryArgs& a, hipStream_t s) {
  if (a.d < 8 || a.d % 8 != 0 || a.d > kQ8RowPer * kWave || a.dq < a.d || a.dq > kQ8RowPer * kWave || a.dq % 128 != 0 ||
      a.nzero < 0 || (a.nzero > 0 && a.zero == nullptr))
    return hipErrorInvalidValue;
  const int64_t per = kBlock / kWave;
  const int64_t grid = (a.nq + per - 1) / per;
  if (grid <= 0 || grid > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(q8_query_kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

}  // namespace cvs
