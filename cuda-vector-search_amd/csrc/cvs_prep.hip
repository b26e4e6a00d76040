// Row preparation: L2 normalisation and zero-padding of fp16 rows in one pass.
//
// Replaces the torch sequences of cuda_vector_search/index.py:35-41
// (_normalize_: fp32 row norm clamped at 1e-12, divide, round to fp16) and
// index.py:27-32 (_pad_width: zero columns up to a multiple of 64), which the
// reference runs on every cosine search for the queries (index.py:89-98, about
// ten small kernels per call) and once over the corpus at Index construction
// (index.py:56-78).
//
// A group of lanes per row: the row is read once in 16-byte pieces (unaligned
// ones where the width or the stride is no multiple of 8), its sum of squares is
// reduced across the group, and the scaled row is written back as fp16 with the
// padding columns zeroed.  Source and destination may be the same rows (the
// group reads its whole row before writing it).  Memory-bound: 2*d bytes read
// and 2*width bytes written per row; 16 lanes a row read 256 consecutive bytes
// per load and keep 3 to 12 loads in flight each.  The sum of squares is in
// fp64 and the scaling a two-float product: fewer instructions than an fp32
// division, and the fp32 quotient is the nearest one whatever the order of the
// sum (an fp32 norm moved one stored element in ~2^14 by an fp16 step).
//
// 500k x 768, normalised: 602 us with one wave a row and 2-byte loads, 266 us
// (5.8 TB/s) so; 300k x 777, padded to 832: 381 -> 184 us.
#include "cvs_common.h"
#include "cvs_kernels.h"

namespace cvs {

namespace {

typedef half8 half8_any __attribute__((aligned(2)));  // 16 bytes at any fp16 address

// LPR lanes per row, P 16-byte pieces per lane: rows of at most 8 * LPR * P
// columns.  P = 0: rows of any width, read twice (sum of squares, then scale and
// write); a lane writes only the columns it read, so in-place rows stay safe.
template <int LPR, int P>
__global__ __launch_bounds__(kBlock) void prep_rows_kernel(PrepArgs a) {
  const int l = threadIdx.x % LPR;
  const int64_t row = (int64_t)blockIdx.x * (kBlock / LPR) + threadIdx.x / LPR;
  if (a.xmax != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *a.xmax = 0.f;
  if (row >= a.n) return;  // a row's lanes stay together
  const _Float16* src = a.src + row * a.src_stride;
  _Float16* dst = a.dst + row * a.dst_width;
  const int full = a.d / 8, tail = a.d % 8;  // whole source pieces, columns of the last, partial one
  const int np = (a.dst_width + 7) / 8;

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
  double ss = 0.;  // the squares are exact in fp32
  auto add = [&](const half8& v) {
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += (double)((float)v[j] * (float)v[j]);
  };
  half8 v[P ? P : 1];
  if constexpr (P > 0) {
#pragma unroll
    for (int i = 0; i < P; ++i) v[i] = piece(i * LPR + l);
#pragma unroll
    for (int i = 0; i < P; ++i) add(v[i]);
  } else if (a.normalize) {
#pragma unroll 4
    for (int c = l; c < np; c += LPR) add(piece(c));
  }
  float inv = 1.f, inv_lo = 0.f;  // 1 / max(||x||, 1e-12) as a sum of two floats
  if (a.normalize) {
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    double r = (double)rsqrtf((float)ss);
    r *= 1.5 - 0.5 * ss * r * r;  // a Newton step: 2^-24 -> 2^-46
    if (ss < 1e-24) r = 1e12;
    if (ss > 1e30) r = 0.;  // an infinite element: the finite ones become 0, as divided by infinity
    inv = (float)r;
    inv_lo = (float)(r - (double)inv);
  }
  // The fp32 number nearest to x / ||x||, then fp16 as the reference rounds.
  auto scaled = [&](_Float16 h) {
#pragma clang fp contract(off)
    const float x = (float)h;
    const float p = x * inv;
    float r = p - fmaf(-x, inv_lo, fmaf(-x, inv, p));  // (keeps the sign of a zero)
    asm("" : "+v"(r));  // rounded to fp32 before fp16 (not a mixed-precision fma), as the reference's quotient
    return (_Float16)r;
  };
  float m = 0.f;  // the stored row's largest magnitude (NaNs skipped)
  auto put = [&](int c, half8 x) {
    if (a.normalize)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = scaled(x[j]);
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
  if constexpr (P > 0) {
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (i * LPR + l < np) put(i * LPR + l, v[i]);
  } else {
#pragma unroll 4
    for (int c = l; c < np; c += LPR) put(c, piece(c));
  }
  if (a.key != nullptr) {  // for the int8 companion's row order
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (l == 0) {
      a.key[row] = __builtin_bit_cast(uint16_t, (_Float16)m);  // m is a half's magnitude: exact
      a.ids[row] = (int)row;
    }
  }
}

template <int LPR, int P>
void launch_lpr(const PrepArgs& a, hipStream_t s) {
  constexpr int rows = kBlock / LPR;
  hipLaunchKernelGGL((prep_rows_kernel<LPR, P>), dim3((unsigned)((a.n + rows - 1) / rows)), dim3(kBlock), 0, s, a);
}

}  // namespace

hipError_t launch_prep(const PrepArgs& a, hipStream_t s) {
  if (a.d < 1 || a.dst_width < a.d || (a.key != nullptr && a.ids == nullptr)) return hipErrorInvalidValue;
  if ((a.n + kBlock / kWave - 1) / (kBlock / kWave) > 0x7fffffff) return hipErrorInvalidValue;
  if (a.dst_width <= 16 * 8 * 3)
    launch_lpr<16, 3>(a, s);
  else if (a.dst_width <= 16 * 8 * 6)
    launch_lpr<16, 6>(a, s);
  else if (a.dst_width <= 16 * 8 * 12)
    launch_lpr<16, 12>(a, s);
  else if (a.dst_width <= 64 * 8 * 8)
    launch_lpr<64, 8>(a, s);
  else
    launch_lpr<64, 0>(a, s);
  return hipGetLastError();
}

}  // namespace cvs
