// Row preparation: L2 normalisation and zero-padding of fp16 rows in one pass.
//
// Replaces the torch sequences of cuda_vector_search/index.py:35-41
// (_normalize_: fp32 row norm clamped at 1e-12, divide, round to fp16) and
// index.py:27-32 (_pad_width: zero columns up to a multiple of 64), which the
// reference runs on every cosine search for the queries (index.py:89-98, about
// ten small kernels per call) and once over the corpus at Index construction
// (index.py:56-78).
//
// 16 lanes per row, two groups of 8: the row is read once in 16-byte pieces
// (unaligned ones where the width or the stride is no multiple of 8), its sum of
// squares is reduced across the lanes, and the scaled row is written back as fp16
// with the padding columns zeroed.  Source and destination may be the same rows
// (a lane writes only what it has read).  Memory-bound: 2*d bytes read and
// 2*width bytes written per row; a row's lanes read 256 consecutive bytes per load
// and keep 1 to 16 loads in flight each.
//
// The stored bits are part of the result, so the arithmetic is fixed: fp32 sums
// over the columns of equal index mod 64, in ascending order, then a tree over
// the 64 sums (32, 16, ... 1 apart), and the fp32 quotient of each element by the
// fp32 norm.  (A norm summed in fp64 moves one stored element in ~2^14 by an fp16
// step, and near neighbours in the results with it.)  8 lanes hold all 64 sums,
// 8 each, and cover 64 columns a load.
//
// 500k x 768, normalised: 595 us with one wave a row and 2-byte loads, 263 us
// (5.8 TB/s) so; 300k x 777, padded to 832: 379 -> 182 us; 200k x 2048 623 -> 302.
#include "cvs_common.h"
#include "cvs_kernels.h"

namespace cvs {

namespace {

typedef half8 half8_any __attribute__((aligned(2)));  // 16 bytes at any fp16 address

constexpr int kGroup = 8;      // lanes that read 64 consecutive columns
constexpr int kRowLanes = 16;  // two such groups a row

// The value in the lane that a DPP control names, within rows of 16 lanes.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// P pieces per lane: rows of at most 128 P columns, whose 64-column steps the two
// groups take in turn (256 consecutive bytes a load).  WIDE: any width, in such
// blocks, read twice (sum of squares, then scale and write).  4 or 5 waves a
// SIMD reach the most (500k x 768: 281 us with 8, 269 with 5; 200k x 2048 312, 302
// with 4), all 8 where a lane has a single load (1M x 100: 113 us, with 5 147).
template <int P, bool WIDE>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(1, P == 1 ? 8 : P <= 6 ? 5 : 4))) void prep_rows_kernel(PrepArgs a) {
  // lane -> piece of 8 columns, so that pieces 4, 2 and 1 apart are a half-row
  // mirror and two quad permutations apart
  const int l = (threadIdx.x ^ (threadIdx.x & 4 ? 3 : 0)) % kGroup;
  const int64_t row = (int64_t)blockIdx.x * (kBlock / kRowLanes) + threadIdx.x / kRowLanes;
  if (a.xmax != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *a.xmax = 0.f;
  if (row >= a.n) return;  // a row's lanes stay together
  const _Float16* src = a.src + row * a.src_stride;
  _Float16* dst = a.dst + row * a.dst_width;
  const int full = a.d / 8, tail = a.d % 8;  // whole source pieces, columns of the last, partial one
  const int np = (a.dst_width + 7) / 8;
  const int c0 = threadIdx.x / kGroup % 2 * kGroup + l;  // this lane's pieces: c0 + i * kRowLanes of every block
  constexpr int kBlockPieces = kRowLanes * P;

  // Source piece c: whole, partial, or zero past the row.  Whole pieces load
  // unconditionally from a clamped index, so that a lane's loads issue together.
  auto piece = [&](int c) {
    half8 v = {};
    if (full > 0) v = *(const half8_any*)(src + 8 * min(c, full - 1));
    if (c >= full) {
      v = half8{};
      if (c == full)
#pragma unroll
        for (int j = 0; j < 7; ++j)
          if (j < tail) v[j] = src[8 * c + j];
    }
    return v;
  };
  half8 v[P];
  auto load = [&](int base) {
#pragma unroll
    for (int i = 0; i < P; ++i) v[i] = piece(base + c0 + i * kRowLanes);
  };
  // sums[j]: of the columns 8 l + j mod 64 (the squares are exact in fp32), in
  // the group whose turn it is; the other one's lanes compute along.
  float sums[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) sums[j] = 0.f;
  auto add_block = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2 * P; ++s) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sums[j] = fmaf((float)v[s / 2][j], (float)v[s / 2][j], sums[j]);
#pragma unroll
      for (int j = 0; j < 8; ++j) sums[j] = dpp<0x128>(sums[j]);  // row_ror:8, to the other group
    }
  };
  float nrm = 1.f, inv = 1.f;
  bool exact = false;  // the quotients need a division
  if (!WIDE) load(0);
  if (a.normalize) {  // x / max(||x||, 1e-12)
    if constexpr (WIDE) {
#pragma unroll 1
      for (int base = 0; base < np; base += kBlockPieces) {
        load(base);
        add_block();
      }
    } else {
      add_block();
    }
    // after the last step (group 1's, handed on) group 0 has the sums
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // 32, 16 and 8 columns apart
      sums[j] += dpp<0x141>(sums[j]);  // row_half_mirror
      sums[j] += dpp<0x4e>(sums[j]);   // quad_perm [2, 3, 0, 1]
      sums[j] += dpp<0xb1>(sums[j]);   // quad_perm [1, 0, 3, 2]
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
#pragma unroll
      for (int j = 0; j < off; ++j) sums[j] += sums[j + off];
    const float other = dpp<0x128>(sums[0]);
    const float ss = threadIdx.x & kGroup ? other : sums[0];
    nrm = fmaxf(sqrtf(ss), 1e-12f);
    inv = 1.f / nrm;
    exact = !__builtin_isfinite(ss);
  }
  // The fp32 number nearest to x / nrm, then fp16.  One remainder step on x * inv
  // reaches it for every x of 11 bits and every nrm of 24 (all 2^33 pairs
  // of significands compared) and keeps the sign of a zero; not with infinities.
  auto scaled = [&](_Float16 h) {
    const float x = (float)h;
    const float p = x * inv;
    float r = fmaf(-fmaf(p, nrm, -x), inv, p);
    asm("" : "+v"(r));  // rounded to fp32 before fp16 (not a mixed-precision fma)
    return (_Float16)r;
  };
  float m = 0.f;  // the stored row's largest magnitude (NaNs skipped)
  auto put = [&](int c, half8 x) {
    if (a.key != nullptr)
#pragma unroll
      for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf((float)x[j]));
    if (8 * c + 8 <= a.dst_width) {
      *(half8_any*)(dst + 8 * c) = x;
    } else {
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (8 * c + j < a.dst_width) dst[8 * c + j] = x[j];
    }
  };
  if (exact) {  // a row with an infinity or a NaN
#pragma unroll 1
    for (int base = 0; base < np; base += kBlockPieces) {
#pragma unroll 1
      for (int i = 0; i < P; ++i) {
        const int c = base + c0 + i * kRowLanes;
        if (c >= np) break;
        half8 x = piece(c);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = (_Float16)((float)x[j] / nrm);
        put(c, x);
      }
    }
  } else {
#pragma unroll 1
    for (int base = 0; base < (WIDE ? np : 1); base += kBlockPieces) {
      if (WIDE) load(base);
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int c = base + c0 + i * kRowLanes;
        if (c < np) {
          half8 x = v[i];
          if (a.normalize)
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = scaled(x[j]);
          put(c, x);
        }
      }
    }
  }
  if (a.key != nullptr) {  // for the int8 companion's row order
#pragma unroll
    for (int off = kRowLanes / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (threadIdx.x % kRowLanes == 0) {
      a.key[row] = __builtin_bit_cast(uint16_t, (_Float16)m);  // m is a half's magnitude: exact
      a.ids[row] = (int)row;
    }
  }
}

template <int P, bool WIDE = false>
void launch_prep_rows(const PrepArgs& a, hipStream_t s) {
  constexpr int rows = kBlock / kRowLanes;
  hipLaunchKernelGGL((prep_rows_kernel<P, WIDE>), dim3((unsigned)((a.n + rows - 1) / rows)), dim3(kBlock), 0, s, a);
}

}  // namespace

hipError_t launch_prep(const PrepArgs& a, hipStream_t s) {
  if (a.d < 1 || a.dst_width < a.d || (a.key != nullptr && a.ids == nullptr)) return hipErrorInvalidValue;
  if ((a.n + kBlock / kWave - 1) / (kBlock / kWave) > 0x7fffffff) return hipErrorInvalidValue;
  if (a.dst_width <= 128)
    launch_prep_rows<1>(a, s);
  else if (a.dst_width <= 128 * 3)
    launch_prep_rows<3>(a, s);
  else if (a.dst_width <= 128 * 6)
    launch_prep_rows<6>(a, s);
  else if (a.dst_width <= 128 * 12)
    launch_prep_rows<12>(a, s);
  else if (a.dst_width <= 128 * 16)
    launch_prep_rows<16>(a, s);
  else
    launch_prep_rows<16, true>(a, s);
  return hipGetLastError();
}

}  // namespace cvs
