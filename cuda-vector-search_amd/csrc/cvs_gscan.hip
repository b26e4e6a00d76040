// Tiled-GEMM scan for large batches: scores query blocks against corpus tiles
// with both operands streamed through LDS, for any width (a multiple of 64).
//
// The query-stationary scan (cvs_scan.hip) holds a wave's queries in registers,
// which limits a wave to 32 queries at width 768 and 16 at 1536: every 1 KiB
// fragment read from LDS then feeds one MFMA, and the LDS, not the matrix cores,
// sets the pace.  Here a wave owns 32 QB queries x 32 RB rows (128 x 128: half a
// fragment read per MFMA) and the width is the loop:
//
//  * 4 waves, 2 query halves x 2 row halves.  A corpus stage is 64 columns of
//    the tile's rows (whole 128-byte lines from HBM), in a ring of 3; the
//    queries, L2-resident, come in phases of 32 columns (two k-steps), in a
//    ring of 3: 144 KB of LDS at 256 x 256, 96 KB of it in flight.
//  * One barrier per phase.  The fragments of a phase's second k-step are
//    consumed after the next phase's barrier, so that the first reads behind a
//    barrier wait under MFMAs.
//  * Accumulators live in AGPRs (256 of them); a tile's epilogue filters as the
//    query-stationary scan does: block maxima against the query's threshold,
//    passing lanes' scores staged in LDS (8 rows an entry), flushed into the
//    wave's candidate lists, full lists cut to their k best.
//
// Measured: 256 x 256 tiles 0.99 PFLOP/s (1000 x 768; 0.93 against 0.90 over
// the whole scan, tail included, of the query-stationary kernel of that width),
// 0.86 at width 1664 where the query-stationary scan reached 0.31, and 128 x
// 128 tiles, two workgroups a CU, 0.76 at width 128 (0.51).
//
// kStore* writes the score matrix from the same tiles, straight from the
// accumulators: lanes swap so that four of them write 64 bytes of a query.
// (32 bytes by two lanes, without the swaps: 1000 x 1024 over 200k rows, 800 MB of
// scores, 523 us in fp32 and 453 in fp16, so 497 and 443.)
#include <type_traits>

#include "cvs_common.h"
#include "cvs_kernels.h"

namespace cvs {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kRing = 3;      // corpus stages and query phases in LDS
constexpr int kStage = 32;    // staged entries per wave
constexpr int kEntry = 8;     // scores of an entry: half of a lane's 16 of a 32 x 32 block

__device__ __forceinline__ constexpr int acc_row(int e) { return 8 * (e >> 2) + (e & 3); }

// c += a x b (ZERO: c = a x b), accumulated in place in AGPRs.  As inline asm:
// with 256 accumulators the compiler's own form moves whole accumulators between
// registers in the loop (305 moves beside 64 MFMAs, or spills).  The operands
// come straight from LDS reads, whose waits the compiler places as usual; the
// caller pads the last results' latency.  Volatile: MFMAs, stage loads and the
// padding stay in the order written.
template <bool ZERO>
__device__ __forceinline__ void mfma_agpr(half8 a, half8 b, f32x16& c) {
  if constexpr (ZERO)
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// 16 bytes per lane from sbase + voff into LDS at lds + 16 * lane (dma16_saddr
// with the default cache policy: other query groups read the same lines).
__device__ __forceinline__ void dma16(uint32_t voff, const void* sbase, uint32_t lds) {
  const uint32_t m = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
  const uint64_t b = (uint64_t)(uintptr_t)sbase;
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  const uint64_t sb = ((uint64_t)hi << 32) | (uint64_t)lo;
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %3\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(m), "v"(voff), "s"(sb)
      : "memory");
}

// wave_compact (cvs_common.h) without LDS scratch: the list's at most kMaxCap
// keys in registers, the k-th best by a bit search over ballots.
__device__ __forceinline__ float wave_compact_regs(float* lv, int* li, int count, int k) {
  constexpr int PER = kMaxCap / kWave;
  const int lane = lane_id();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // the wave's own stores to the list, read back past the vector L1
  uint64_t key[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int p = j * kWave + lane;
    key[j] = p < count ? make_key(coherent_load(lv + p), coherent_load(li + p)) : 0ull;
  }
  uint64_t t = 0;  // the largest t with #(keys >= t) >= k
#pragma unroll 1
  for (int bit = 63; bit >= 0; --bit) {
    const uint64_t cand = t | (1ull << bit);
    int c = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) c += __popcll(__ballot(key[j] >= cand));
    if (c >= k) t = cand;
  }
  int base = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint64_t mk = __ballot(key[j] >= t);
    if (key[j] >= t) {
      const int p = base + lanes_below(mk);
      lv[p] = key_score(key[j]);
      li[p] = key_id(key[j]);
    }
    base += __popcll(mk);
  }
  wait_vmcnt<0>();
  return key_score(t);
}

// Two scores as fp16.
__device__ __forceinline__ uint32_t pack2(float x, float y) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, half2v{(_Float16)x, (_Float16)y});
}

// The N scores v of rows row, row + 1, ... below n into a query's scores `out`
// (16 bytes at the element's alignment: n may be odd).
template <int N, class T, class V>
__device__ __forceinline__ void store_rows(T* out, int64_t row, int64_t n, V v) {
  typedef V any __attribute__((aligned(sizeof(T))));
  if (row + N <= n) {
    *reinterpret_cast<any*>(out + row) = v;
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (row + j < n) out[row + j] = v[j];
  }
}

template <int QB, int RB, int MODE>
__global__ __launch_bounds__(kBlock, QB * RB > 4 ? 1 : 2) void gscan_kernel(ScanArgs a) {
  constexpr int TQ = 64 * QB, TR = 64 * RB;   // queries, rows per workgroup tile
  constexpr int LA = TR / 32, LQ = TQ / 64;   // 1 KiB loads per wave: of a corpus stage, of a query phase
  constexpr int ASTAGE = TR * 128, QPHASE = TQ * 64;
  constexpr bool APP = MODE == kAppend;
  constexpr bool STORE = MODE == kStoreF32 || MODE == kStoreF16;
  static_assert(APP || STORE || MODE == kMax, "append, sampling and the score matrix");
  __shared__ __attribute__((aligned(1024))) unsigned char sa[kRing * ASTAGE];
  __shared__ __attribute__((aligned(1024))) unsigned char sq[kRing * QPHASE];
  __shared__ int lcnt[APP ? 2 : 1][APP ? TQ : 1];     // entries in each owned list
  __shared__ float thr_s[APP ? 2 : 1][APP ? TQ : 1];  // per-query filter threshold
  __shared__ __attribute__((aligned(16))) float st_val[APP ? 4 : 1][APP ? kStage * kEntry : 4];
  __shared__ int st_meta[APP ? 4 : 1][APP ? 2 * kStage : 1];  // (query, first row)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wq = w & 1, wr = w >> 1;
  const int col = lane & 31, kg = lane >> 5;

  int grp, chunk;
  {
    const int id = blockIdx.x;
    if (a.xcd_pair) {  // a chunk's query groups on one XCD: its rows come from HBM once
      const int slot = id >> 3;
      grp = slot % a.groups;
      chunk = (slot / a.groups) * 8 + (id & 7);
    } else {
      grp = id % a.groups;
      chunk = id / a.groups;
    }
  }
  int64_t t_begin, t_end;
  if (MODE == kMax) {  // spt consecutive tiles centred on an evenly spread position
    const int64_t centre = ((2 * (int64_t)chunk + 1) * a.ntiles) / (2 * (int64_t)a.nsample);
    t_begin = centre - a.spt / 2;
    if (t_begin > a.ntiles - a.spt) t_begin = a.ntiles - a.spt;
    if (t_begin < 0) t_begin = 0;
    t_end = t_begin + a.spt;
  } else {
    t_begin = (int64_t)chunk * a.tpc;
    t_end = t_begin + a.tpc < a.ntiles ? t_begin + a.tpc : a.ntiles;
  }
  const int d = a.d;
  const int64_t n = a.n;
  const int nc = d >> 6;  // stages per tile
  const int q0 = grp * TQ;

  // ---- loads.  Corpus stage: row R of the tile at R * 128, slot s holding piece
  // s ^ piece_swz(R).  Query phase: line L holds the 64 bytes of queries 2 L and
  // 2 L + 1, slot s piece p = s ^ ((L >> 1) & 3) (query 2 L + p / 4, its piece
  // p % 4).  Either way 16 consecutive rows' equal pieces, what the lanes of a
  // fragment read together, lie on distinct banks.
  uint32_t voa[LA], voq[LQ];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int R = (w + 4 * j) * 8 + (lane >> 3);
    voa[j] = (uint32_t)R * (uint32_t)(2 * d) + (((lane & 7) ^ piece_swz(R)) << 4);
  }
#pragma unroll
  for (int j = 0; j < LQ; ++j) {
    const int L = (w + 4 * j) * 8 + (lane >> 3);
    const int p = (lane & 7) ^ ((L >> 1) & 3);
    const int ql = min(2 * L + (p >> 2), a.nq - 1 - q0);  // past the batch: the last query again
    voq[j] = (uint32_t)ql * (uint32_t)(2 * d) + ((p & 3) << 4);
  }
  const uint32_t la0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)sa);
  const uint32_t lq0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)sq);
  // Issue cursors: past the last tile the last one again, so that every wave
  // always counts the same loads; rows past n: the last row again.
  const unsigned char* qbase = reinterpret_cast<const unsigned char*>(a.q + (int64_t)q0 * d);
  const unsigned char* abase;
  int64_t it_t = min(t_begin, a.ntiles - 1);
  int it_c = 0, ia = 0, it_p = 0, iq = 0;
  auto enter_tile = [&]() {
    abase = reinterpret_cast<const unsigned char*>(a.x) + it_t * TR * (2 * (int64_t)d);
    if ((it_t + 1) * TR > n) {
      const int last = (int)(n - 1 - it_t * TR);
#pragma unroll
      for (int j = 0; j < LA; ++j) {
        const int R = (w + 4 * j) * 8 + (lane >> 3);
        voa[j] = (uint32_t)min(R, last) * (uint32_t)(2 * d) + (((lane & 7) ^ piece_swz(R)) << 4);
      }
    }
  };
  enter_tile();
  auto load_a = [&](int j) { dma16(voa[j], abase, la0 + (uint32_t)(ia * ASTAGE + w * 1024 + j * 4096)); };
  auto load_q = [&](int j) { dma16(voq[j], qbase + it_p * 64, lq0 + (uint32_t)(iq * QPHASE + w * 1024 + j * 4096)); };
  auto next_a = [&]() {
    abase += 128;
    if (++it_c == nc) {
      it_c = 0;
      if (it_t + 1 < a.ntiles) ++it_t;
      enter_tile();
    }
    if (++ia == kRing) ia = 0;
  };
  auto next_q = [&]() {
    if (++it_p == 2 * nc) it_p = 0;
    if (++iq == kRing) iq = 0;
  };
  auto issue_a = [&]() {
#pragma unroll
    for (int j = 0; j < LA; ++j) load_a(j);
    next_a();
  };
  auto issue_q = [&]() {
#pragma unroll
    for (int j = 0; j < LQ; ++j) load_q(j);
    next_q();
  };
  issue_a();

  float thr[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qi = q0 + (wq * QB + qb) * 32 + col;
    thr[qb] = qi >= a.nq ? kNoThreshold : (APP && a.tau ? a.tau[qi] : -__builtin_inff());
  }
  if constexpr (APP) {
    for (int i = tid; i < 2 * TQ; i += kBlock) {
      (&lcnt[0][0])[i] = 0;
      const int qi = q0 + i % TQ;
      (&thr_s[0][0])[i] = qi >= a.nq ? kNoThreshold : (a.tau ? a.tau[qi] : -__builtin_inff());
    }
  }
  wait_vmcnt<0>();  // retires the threshold loads: the compiler then waits on no vector load inside the loop
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) asm volatile("" : "+v"(thr[qb]));
  issue_q();
  issue_a();
  issue_q();

  // ---- fragments
  int aoff[4], boff[2];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) aoff[kk] = (wr * RB * 32 + col) * 128 + (((2 * kk + kg) ^ piece_swz(col)) << 4);
#pragma unroll
  for (int j = 0; j < 2; ++j)
    boff[j] = ((wq * QB * 32 + col) >> 1) * 128 + ((((col & 1) * 4 + 2 * j + kg) ^ ((col >> 2) & 3)) << 4);
  half8 fa0[RB], fb0[QB], fa1[RB], fb1[QB];
  int ca = 0, cq = 0;  // ring slots of the current stage and phase
  auto read_frags = [&](int kk, half8 (&fa)[RB], half8 (&fb)[QB]) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) fa[rb] = *(const half8*)(sa + ca * ASTAGE + aoff[kk] + rb * 4096);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) fb[qb] = *(const half8*)(sq + cq * QPHASE + boff[kk & 1] + qb * 2048);
  };
  f32x16 acc[RB][QB];
  // The MFMAs of one k-step, side(i) between the i-th and the next.
  auto mfma = [&](auto first, const half8 (&fa)[RB], const half8 (&fb)[QB], auto side) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        mfma_agpr<decltype(first)::value>(fa[rb], fb[qb], acc[rb][qb]);
        side(rb * QB + qb);
      }
  };
  auto nothing = [](int) {};

  // ---- candidates
  int st_n = 0;  // wave-uniform count of staged entries
  auto flush = [&]() {  // two lanes per entry, 4 scores each
    const int list = chunk * 2 + wr;
    const int er = lane >> 1;
    const bool have = er < st_n;
    const int ql = have ? st_meta[w][2 * er] : 0;
    const int rbase = (have ? st_meta[w][2 * er + 1] : 0) + 8 * (lane & 1);
    const f32x4 ev = *(const f32x4*)(&st_val[w][(have ? er : 0) * kEntry + 4 * (lane & 1)]);
    const int64_t lbase = ((int64_t)(q0 + ql) * a.nlists + list) * a.cap;
    unsigned todo = 0;
    if (have) {
      const float tq = thr_s[wr][ql];
#pragma unroll
      for (int e = 0; e < 4; ++e) todo |= (ev[e] >= tq && rbase + e < n ? 1u : 0u) << e;
    }
#pragma unroll 1
    while (true) {
      const int cnt = __popc(todo);
      const int pos = cnt ? atomicAdd(&lcnt[wr][ql], cnt) : 0;
      const int room = a.cap - pos;
      int put = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (((todo >> e) & 1u) && put < room) {
          a.lv[lbase + pos + put] = ev[e];
          a.li[lbase + pos + put] = rbase + e;
          todo &= ~(1u << e);
          ++put;
        }
      }
      uint64_t om = __ballot(todo != 0);
      if (!om) break;
      // lists that filled: cut to their k best, then the scores left are tried again
#pragma unroll 1
      while (om) {
        const int ql0 = __shfl(ql, __ffsll((unsigned long long)om) - 1);
        const int64_t base0 = ((int64_t)(q0 + ql0) * a.nlists + list) * a.cap;
        const float prev = thr_s[wr][ql0];
        const float nt = fmaxf(prev, wave_compact_regs(a.lv + base0, a.li + base0, a.cap, a.k));
        if (lane == 0) {
          lcnt[wr][ql0] = a.k;
          thr_s[wr][ql0] = nt;
        }
        om &= ~__ballot(ql == ql0);
      }
      if (todo) {
        const float tq = thr_s[wr][ql];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ev[e] < tq) todo &= ~(1u << e);
      }
    }
    st_n = 0;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) thr[qb] = thr_s[wr][(wq * QB + qb) * 32 + col];
  };

  float umx[MODE == kMax ? RB : 1][MODE == kMax ? QB : 1];  // kMax, agg: maxima over all sampled tiles
  if constexpr (MODE == kMax) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) umx[rb][qb] = -__builtin_inff();
  }

#pragma unroll 1
  for (int64_t t = t_begin; t < t_end; ++t) {
    // One stage, two phases.  A phase (and its stage) has landed for every wave
    // behind its barrier, and the ring slots read before it are free for the
    // loads issued there; in issue order, one stage's and one phase's loads
    // follow those that this phase needs.  The loads go between MFMAs, whose
    // 32 cycles each leave room to issue them.
    auto stage = [&](auto first) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        wait_vmcnt_lgkm0<LA + LQ>();
        __builtin_amdgcn_s_barrier();
        read_frags(2 * h, fa0, fb0);
        if (h == 0 && decltype(first)::value) {
          issue_q();
          issue_a();
        } else {
          mfma(std::false_type{}, fa1, fb1, [&](int i) {
            if (i < LQ) load_q(i);
            else if (h == 0 && i < LQ + LA) load_a(i - LQ);
          });
          static_assert(LQ + LA <= RB * QB || RB * QB <= 8, "a load per MFMA");
          if constexpr (RB * QB < LQ + LA) {  // (the smaller tiles have fewer MFMAs than loads)
#pragma unroll
            for (int i = RB * QB; i < LQ + LA; ++i)
              if (h == 0) load_a(i - LQ);
          }
          next_q();
          if (h == 0) next_a();
        }
        read_frags(2 * h + 1, fa1, fb1);
        if (h == 0) mfma(first, fa0, fb0, nothing);
        else mfma(std::false_type{}, fa0, fb0, nothing);
        if (++cq == kRing) cq = 0;
      }
      if (++ca == kRing) ca = 0;
    };
    stage(std::true_type{});
#pragma unroll 1
    for (int c = 1; c < nc; ++c) stage(std::false_type{});
    mfma(std::false_type{}, fa1, fb1, nothing);
    // the last results' latency (as pad_mfma_result), and every read of them behind it
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+a"(acc[RB - 1][QB - 1]));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) asm volatile("" : "+a"(acc[rb][qb]));

    // ---- epilogue: acc[rb][qb][e] = score(query (wq QB + qb) 32 + col,
    //                 row rowb + 32 rb + acc_row(e)).  Rows past n repeat the last
    // row: the flush drops them, and a sampling unit that holds one is left out.
    const int64_t rowb = t * TR + wr * RB * 32 + 4 * kg;
    if constexpr (MODE == kMax) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const int qi = q0 + (wq * QB + qb) * 32 + col;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          float m = acc[rb][qb][0];
#pragma unroll
          for (int e = 1; e < 16; ++e) m = fmaxf(m, acc[rb][qb][e]);
          if (rowb + rb * 32 + acc_row(15) >= n) m = -__builtin_inff();
          if (a.agg)
            umx[rb][qb] = fmaxf(umx[rb][qb], m);
          else if (qi < a.nq)
            a.umax[(int64_t)qi * a.units + ((chunk * a.spt + (t - t_begin)) * 2 + wr) * (2 * RB) + 2 * rb + kg] = m;
        }
      }
    } else if constexpr (STORE) {
      // Lanes of 16 swap halves of the block, so that 4 lanes write 64 bytes of a
      // query at once: afterwards a lane holds queries h * 16 + col % 16, h = 0, 1.
      const int qcol = q0 + wq * QB * 32 + (col & 15);
      const int up = col >> 4;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          asm volatile("" : "+a"(acc[rb][qb]));  // keeps the block's reads here (all 256 would not fit)
          const f32x16 c = acc[rb][qb];
          if constexpr (MODE == kStoreF32) {
#pragma unroll
            for (int g = 0; g < 4; g += 2) {  // rows 8 g + 4 kg + 0..3, and 8 more
              f32x4 v[2];
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(c[4 * g + j]),
                                                                __float_as_uint(c[4 * g + 4 + j]), false, false);
                v[0][j] = __uint_as_float(r[0]);
                v[1][j] = __uint_as_float(r[1]);
              }
              const int64_t row = rowb + 32 * rb + 8 * (g + up);
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const int qi = qcol + 32 * qb + 16 * h;
                if (qi < a.nq) store_rows<4>(static_cast<float*>(a.out) + (int64_t)qi * n, row, n, v[h]);
              }
            }
          } else {
            uint4v v[2];  // rows 16 p + 8 kg + 0..7: the halves' fours swapped
#pragma unroll
            for (int p = 0; p < 2; ++p) {
#pragma unroll
              for (int j = 0; j < 2; ++j) {
                const auto r = __builtin_amdgcn_permlane32_swap(pack2(c[8 * p + 2 * j], c[8 * p + 2 * j + 1]),
                                                                pack2(c[8 * p + 4 + 2 * j], c[8 * p + 5 + 2 * j]), false, false);
                v[p][j] = r[0];
                v[p][2 + j] = r[1];
              }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const auto r = __builtin_amdgcn_permlane16_swap(v[0][j], v[1][j], false, false);
              v[0][j] = r[0];
              v[1][j] = r[1];
            }
            const int64_t row = rowb - 4 * kg + 32 * rb + 16 * up + 8 * kg;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int qi = qcol + 32 * qb + 16 * h;
              if (qi < a.nq)
                store_rows<8>(static_cast<_Float16*>(a.out) + (int64_t)qi * n, row, n, __builtin_bit_cast(half8, v[h]));
            }
          }
        }
      }
    } else {
      // Stages the passing lanes' scores of half blocks b0, b0 + 1, ... (of half
      // block b0 those of the lanes in `rem`) until the staging area is full
      // (true: flush and call again) or the tile is done.
      int b0 = 0;
      uint64_t rem = ~0ull;
      auto stage_tile = [&]() -> bool {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            asm volatile("" : "+a"(acc[rb][qb]));  // keeps the block's reads here (all 256 would not fit)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int b = (qb * RB + rb) * 2 + h;
              if (b < b0) continue;
              float m = acc[rb][qb][8 * h];
#pragma unroll
              for (int e = 1; e < 8; ++e) m = fmaxf(m, acc[rb][qb][8 * h + e]);
              const uint64_t mk = __ballot(m >= thr[qb]) & rem;
              rem = ~0ull;
              if (mk == 0) continue;
              const int p = st_n + lanes_below(mk);
              const bool mine = (mk >> lane) & 1;
              if (mine && p < kStage) {
#pragma unroll
                for (int e = 0; e < 8; e += 4)
                  *(f32x4*)(&st_val[w][p * kEntry + e]) =
                      f32x4{acc[rb][qb][8 * h + e], acc[rb][qb][8 * h + e + 1], acc[rb][qb][8 * h + e + 2],
                            acc[rb][qb][8 * h + e + 3]};
                st_meta[w][2 * p] = (wq * QB + qb) * 32 + col;
                st_meta[w][2 * p + 1] = (int)rowb + rb * 32 + 16 * h;
              }
              st_n += __popcll(mk);
              if (st_n > kStage) {
                rem = __ballot(mine && p >= kStage);
                b0 = b;
                st_n = kStage;
                return true;
              }
            }
          }
        }
        return false;
      };
      while (stage_tile()) flush();
    }
  }
  if constexpr (APP) {
    if (st_n > 0) flush();
    // The lists of a few queries that stayed half full (scores that tie by the
    // thousand, as a query of zeros has) are cut to their k best where that takes
    // most of them away: the select reads all lists of a query in one workgroup
    // (64 x 512 over 100k rows, k = 10, with one query of zeros: 398 us, 252 with the
    // query-stationary scan's fewer lists, so 131; with 8 405, 312 and 225).  Where
    // most queries have such lists their selects run side by side, and the cuts
    // would not (rows stored by ascending score 53 us, every list cut 127).
#pragma unroll 1
    for (int i = 0; i < 32 * QB; i += kWave) {
      const int ql = wq * QB * 32 + i + lane;
      const int c = i + lane < 32 * QB ? lcnt[wr][ql] : 0;
      uint64_t om = __ballot(2 * c >= a.cap && c >= 4 * a.k);
      if (__popcll(om) > 8) om = 0;
#pragma unroll 1
      while (om) {
        const int l = __ffsll((unsigned long long)om) - 1;
        const int ql0 = wq * QB * 32 + i + l;
        const int64_t base0 = ((int64_t)(q0 + ql0) * a.nlists + chunk * 2 + wr) * a.cap;
        wave_compact_regs(a.lv + base0, a.li + base0, __shfl(c, l), a.k);
        if (lane == 0) lcnt[wr][ql0] = a.k;
        om &= om - 1;
      }
    }
  } else if (MODE == kMax && a.agg) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int qi = q0 + (wq * QB + qb) * 32 + col;
      if (qi < a.nq)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          a.umax[(int64_t)qi * a.units + (chunk * 2 + wr) * (2 * RB) + 2 * rb + kg] = umx[MODE == kMax ? rb : 0][MODE == kMax ? qb : 0];
    }
  }
  // the trailing loads land before this workgroup's LDS can be handed on; counts are final
  wait_vmcnt_lgkm0<0>();
  __builtin_amdgcn_s_barrier();
  if constexpr (APP) {
    for (int i = tid; i < 2 * TQ; i += kBlock) {
      const int qi = q0 + i % TQ;
      if (qi < a.nq) a.lcount[(int64_t)qi * a.nlists + chunk * 2 + i / TQ] = (&lcnt[0][0])[i];
    }
  }
}

template <int QB, int RB>
hipError_t launch_g(int mode, const ScanArgs& a, int grid, hipStream_t s) {
  if (mode == kAppend)
    hipLaunchKernelGGL((gscan_kernel<QB, RB, kAppend>), dim3(grid), dim3(kBlock), 0, s, a);
  else if (mode == kStoreF32)
    hipLaunchKernelGGL((gscan_kernel<QB, RB, kStoreF32>), dim3(grid), dim3(kBlock), 0, s, a);
  else if (mode == kStoreF16)
    hipLaunchKernelGGL((gscan_kernel<QB, RB, kStoreF16>), dim3(grid), dim3(kBlock), 0, s, a);
  else if constexpr (RB == 2)  // sampling: the smallest tiles of a batch only
    hipLaunchKernelGGL((gscan_kernel<QB, RB, kMax>), dim3(grid), dim3(kBlock), 0, s, a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gscan(const ScanCfg& c, int mode, const ScanArgs& a, int grid, hipStream_t s) {
  const bool store = mode == kStoreF32 || mode == kStoreF16;
  if ((mode != kAppend && mode != kMax && !store) || (store && a.out == nullptr) || a.d < 64 || a.d % 64 != 0 || a.d > kGscanMaxWidth || a.nq < 1 || a.ntiles < 1 ||
      a.umax_in != nullptr || a.qq_out != nullptr || (mode == kMax && (a.umax == nullptr || a.agg > 1)) ||
      (mode == kAppend && (a.cap > kMaxCap || a.k > a.cap || a.nlists != a.nchunks * 2)))
    return hipErrorInvalidValue;
  if (c.qb == 4 && c.rb == 4) return launch_g<4, 4>(mode, a, grid, s);
  if (c.qb == 2 && c.rb == 4) return launch_g<2, 4>(mode, a, grid, s);
  if (c.qb == 2 && c.rb == 2) return launch_g<2, 2>(mode, a, grid, s);
  if (c.qb == 1 && c.rb == 4) return launch_g<1, 4>(mode, a, grid, s);
  if (c.qb == 1 && c.rb == 2) return launch_g<1, 2>(mode, a, grid, s);
  return hipErrorInvalidValue;
}

}  // namespace cvs
