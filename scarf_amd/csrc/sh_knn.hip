// Exact k-nearest-neighbour search (squared L2) on MFMA with an error-bounded
// low-precision screen.  Replaces scarf's hnswlib index (ann.py:14-28, 194-205,
// 290-326) and fix_knn_query (ann.py:31-52).
//
// The screen (MFMA tiles, threshold filter, candidate buffers) and the threshold pass are
// in sh_knn_screen.h; this file packs the operands, merges and re-ranks the candidates.
#include <float.h>

#include <algorithm>
#include <cmath>

#include "sh_knn_screen.h"

namespace sh {

__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

int32_t pack_k(int dtype, int32_t D) {
  if (dtype == SH_F32) return (int32_t)align_up((size_t)D + 1, 8);
  if (dtype == SH_BF16) return (int32_t)align_up((size_t)D + 3, 16);
  if (dtype == SH_FP8) return (int32_t)align_up((size_t)D, 64);
  return -1;
}

// Bytes per packed row: K operand elements, plus (FP8) a 16-byte trailer holding the
// row's ||r||^2 (f32) and its E8M0 scale exponent (biased, i32).
int64_t pack_row_bytes(int dtype, int32_t D) {
  const int32_t K = pack_k(dtype, D);
  if (K < 0) return -1;
  if (dtype == SH_F32) return (int64_t)K * 4;
  if (dtype == SH_BF16) return (int64_t)K * 2;
  return (int64_t)K + 16;
}

// ---------------------------------------------------------------------------------
// Packing, `rb` rows per workgroup staged through LDS: the FP32 rows are read coalesced with
// several loads in flight, one thread per row sums the squared norm in feature order (FP64,
// the value that the BF16 split needs) and, for FP8, finds the row's scale, and all threads
// then write the packed rows as consecutive 32-bit words.  With a thread per row throughout,
// every access touched a line per lane: 1.5M FP8 rows of 100 took 4.4 ms (now 187 us),
// 1M BF16 rows of 50 313 us (now 105).
//
// FP32: [r, ||r||^2, 0...] / [-2q, 1, 0...].  BF16: the norm as an unevaluated sum of three
// bf16 values (24 significant bits).  FP8: x / 2^e in OCP E4M3 (the converter rounds to
// nearest even; values are clamped to its +-448) with e the smallest power of two that
// brings max|x| under 448, and a trailer of the norm and e.
constexpr int kPackThreads = 256;
constexpr int kPackRows = 64;  // at most

// Smallest e with |amax| / 2^e <= 448, clamped to the E8M0 range (an infinite amax too).
__device__ __forceinline__ int fp8_exp(float amax) {
  if (!(amax > 0.f)) return 0;
  int ex = (int)fminf(fmaxf(ceilf(log2f(amax / 448.0f)), -126.f), 126.f);
  while (ex < 126 && ldexpf(amax, -ex) > 448.0f) ++ex;
  return ex;
}

template <int DT>
__global__ void __launch_bounds__(kPackThreads) k_pack(const float *__restrict__ E, int64_t n,
                                                       int32_t D, int64_t lde, int role,
                                                       int32_t K, int rb,
                                                       uint32_t *__restrict__ out,
                                                       float *__restrict__ aux) {
  extern __shared__ float pack_lds[];  // [rb][D | 1]
  __shared__ double s_n2[kPackRows];
  __shared__ int s_ex[kPackRows];
  const int tid = threadIdx.x, ld = D | 1;
  const int64_t r0 = (int64_t)blockIdx.x * rb;
  const int rows = (int)min<int64_t>(rb, n - r0);
  const float *src = E + r0 * lde;
#pragma unroll 4
  for (int e = tid; e < rows * D; e += kPackThreads) {
    const int r = e / D, t = e - r * D;
    pack_lds[r * ld + t] = src[r * lde + t];
  }
  __syncthreads();
  if (tid < rows) {
    const float *x = pack_lds + tid * ld;
    double s = 0.0;
    float amax = 0.f;
#pragma unroll 4
    for (int t = 0; t < D; ++t) {
      s += (double)x[t] * (double)x[t];
      if (DT == SH_FP8) amax = fmaxf(amax, fabsf(role == 0 ? x[t] : 2.0f * x[t]));
    }
    s_n2[tid] = s;
    if (DT == SH_FP8) s_ex[tid] = fp8_exp(amax);
    if (aux) aux[r0 + tid] = (float)s;
  }
  __syncthreads();
  const int words = DT == SH_F32 ? K : DT == SH_BF16 ? K / 2 : K / 4 + 4;  // per row
  for (int e = tid; e < rows * words; e += kPackThreads) {
    const int r = e / words, wd = e - r * words;
    const float *x = pack_lds + r * ld;
    uint32_t o = 0;
    if (DT == SH_F32) {
      o = __float_as_uint(wd < D    ? (role == 0 ? x[wd] : -2.0f * x[wd])
                          : wd == D ? (role == 0 ? (float)s_n2[r] : 1.0f)
                                    : 0.f);
    } else if (DT == SH_BF16) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int t = 2 * wd + u;
        uint16_t b = 0;
        if (t < D) {
          b = f2bf(role == 0 ? x[t] : -2.0f * x[t]);
        } else if (t < D + 3) {
          if (role == 0) {
            const double s = s_n2[r];
            const float hi = bf2f(f2bf((float)s));
            const double r1 = s - (double)hi;
            const float mid = bf2f(f2bf((float)r1));
            const float lo = bf2f(f2bf((float)(r1 - (double)mid)));
            b = f2bf(t == D ? hi : t == D + 1 ? mid : lo);
          } else {
            b = f2bf(1.0f);
          }
        }
        o |= (uint32_t)b << (16 * u);
      }
    } else if (wd < K / 4) {
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = 4 * wd + u;
        const float y = t < D ? ldexpf(role == 0 ? x[t] : -2.0f * x[t], -s_ex[r]) : 0.f;
        v[u] = fminf(fmaxf(y, -448.f), 448.f);
      }
      int p = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
      p = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], p, true);
      o = (uint32_t)p;
    } else if (wd == K / 4) {
      o = __float_as_uint(role == 0 ? (float)s_n2[r] : 0.f);
    } else if (wd == K / 4 + 1) {
      o = (uint32_t)(s_ex[r] + 127);  // E8M0 biased exponent
    }
    out[r0 * words + e] = o;
  }
}


// A query's starting threshold from the threshold pass: the rank-th smallest of its `m`
// slot minima (k_bound), one wave per query.  The orderable images are searched bit by bit
// from the top (count the values at or below a prefix); the low kTauSkip bits are left set,
// which only raises the threshold.  Fewer than `rank` finite minima leave it open.
constexpr int kTauSkip = 4;
constexpr int kTauSlots = 64 * 32;  // at most
// Wave sum with DPP lane moves, the same value in every lane.
__device__ __forceinline__ int wave_sum_i32(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);   // lane ^ 1
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);   // lane ^ 2
  v += __builtin_amdgcn_update_dpp(0, v, 0x124, 0xF, 0xF, true);  // row_ror:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, true);  // row_ror:8
  return (__builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16)) +
         (__builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48));
}
// Wave or, likewise.
__device__ __forceinline__ uint32_t wave_or_u32(uint32_t x) {
  int v = (int)x;
  v |= __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);
  v |= __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);
  v |= __builtin_amdgcn_update_dpp(0, v, 0x124, 0xF, 0xF, true);
  v |= __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, true);
  return (uint32_t)((__builtin_amdgcn_readlane(v, 0) | __builtin_amdgcn_readlane(v, 16)) |
                    (__builtin_amdgcn_readlane(v, 32) | __builtin_amdgcn_readlane(v, 48)));
}
// How many of a wave's E predicates per lane hold.  LANES: every lane counts its own and one
// wave sum follows, the shorter chain of a wave that works alone; else a ballot and a scalar
// popcount each, which take fewer vector instructions where many waves share a SIMD (the
// thresholds of a million queries 427 against 656 us).
template <bool LANES, int E, class P>
__device__ __forceinline__ int wave_count(P pred) {
  int c = 0;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    if constexpr (LANES)
      c += pred(i);
    else
      c += __popcll(__builtin_amdgcn_ballot_w64(pred(i)));
  }
  if constexpr (LANES) c = wave_sum_i32(c);
  return c;
}

template <int EL>
__global__ void __launch_bounds__(256) k_tau(const float *__restrict__ slot_min, int64_t nq,
                                             int m, int rank, float *__restrict__ tau0,
                                             int32_t *__restrict__ zero) {
  const int lane = threadIdx.x & 63;
  if (zero && blockIdx.x == 0 && threadIdx.x == 0) *zero = 0;
  const int64_t q = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= nq) return;
  uint32_t v[EL];
#pragma unroll
  for (int i = 0; i < EL; ++i) {
    const int e = i * 64 + lane;
    v[i] = e < m ? float_ord(slot_min[q * m + e]) : 0xffffffffu;
  }
  uint32_t prefix = 0;
  for (int bit = 31; bit >= kTauSkip; --bit) {
    const uint32_t t = prefix | ((1u << bit) - 1u);
    const int below = wave_count<(EL >= 8), EL>([&](int i) { return v[i] <= t; });
    if (below < rank) prefix |= 1u << bit;
  }
  const uint32_t t = prefix | ((1u << kTauSkip) - 1u);
  if (lane == 0) {
    float tau = kOpen;
    if (t < float_ord(kOpen)) {
      const float x = ord_float(t);
      tau = fminf(x + fabsf(x) * 0x1p-16f, kOpen);
    }
    tau0[q] = tau;
  }
}

// Best `pool` keys of each query over the segments that a sliced scan left in its buffers
// (two halves per slice, counts in seg_cnt), sorted.  One wave per query.  The counts are
// scanned into offsets in LDS and every lane finds its keys' segments by bisection, so the
// loads are independent whatever the counts.  64 * E keys are taken at a time (the usual
// query has fewer): the pool-th smallest is searched bit by bit on the keys' distance half
// (count what lies at or below a prefix; on the index half too where distances tie), the
// keys up to it are packed together in LDS, and only they are sorted: at a million queries
// of about 240 keys, half the time of sorting them all.  The search starts below the bits that
// all keys share and ends once a count is the pool, some ten rounds instead of 32: 2.41 ->
// 1.75 ms at a million queries, 228 -> 168 us at 100,000, 14.6 -> 11.8 for one.  (The same in
// k_tau, whose values end alike less often, took 536 us instead of 426 at a million.)
//
// BITS: the segments hold plain float bits above the index (k_collect), not make_key's word.
// fail (or NULL): queries whose keys are incomplete -- a segment that overflowed, or fewer
// than `need` keys -- are listed there instead, to be screened again, and so are those with more
// keys than kMergeRounds times 64 * E (ties spread evenly over many slices): one wave takes 19 us
// for each such part, and screening 1000 queries again 0.6 to 1.8 ms.  1000 queries x 300,000,
// half of both one row: 6.9 ms with no limit, 1.3 with one; ties of 15,000 in 0.77 and, were
// they screened again, 1.49 ms.
// list (or NULL): positions list_base.. of a list of queries whose length the device knows.
constexpr int kMergeRounds = 96;
template <int PE, int E, bool BITS>
__global__ void __launch_bounds__(256) k_pool_merge(
    const uint64_t *__restrict__ buf, const int32_t *__restrict__ seg_cnt, int64_t n, int S,
    int cap, int pool, int need, const int32_t *__restrict__ list,
    const int32_t *__restrict__ list_n, int32_t list_base, int32_t *__restrict__ fail,
    int32_t *__restrict__ fail_n, int32_t fail_base, uint64_t *__restrict__ out,
    int32_t *__restrict__ out_cnt) {
  extern __shared__ uint64_t merge_lds[];  // [4][pool] keys, then [4][2 S] offsets
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t p = (int64_t)blockIdx.x * 4 + w;
  if (list) n = min(n, (int64_t)*list_n - list_base);
  if (p >= n) return;
  const int ns = 2 * S, room = cap / 2;
  uint64_t *kept = merge_lds + w * pool;
  int *off = reinterpret_cast<int *>(merge_lds + 4 * pool) + w * ns;
  // a lane takes a run of consecutive segments: independent loads, one scan over the lanes
  const int run = (ns + 63) / 64;
  int mine = 0;
  bool over = false;
  for (int i = 0; i < run; ++i) {
    const int sg = lane * run + i;
    const int c = sg < ns ? seg_cnt[p * ns + sg] : 0;
    over |= c > room;
    if (sg < ns) off[sg] = mine;
    mine += c;
  }
  int inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(inc, o, kWave);
    if (lane >= o) inc += up;
  }
  const int total = __shfl(inc, 63, kWave);
  for (int i = 0; i < run; ++i) {
    const int sg = lane * run + i;
    if (sg < ns) off[sg] += inc - mine;
  }
  if (fail && (wave_any(over) || total < need || total > kMergeRounds * 64 * E)) {
    if (lane == 0) fail[atomicAdd(fail_n, 1)] = fail_base + (int32_t)p;
    return;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  int have = 0, next = 0;  // keys kept in LDS, keys taken in
  do {
    uint64_t v[E];
    const int fresh = min(total - next, 64 * E - have);
    const int m = have + fresh;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int e = i * 64 + lane;
      v[i] = ~0ull;
      if (e < have) {
        v[i] = kept[e];
      } else if (e < m) {
        const int src = next + (e - have);
        int lo = 0, hi = ns - 1;  // last segment whose offset is <= src
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (off[mid] <= src)
            lo = mid;
          else
            hi = mid - 1;
        }
        v[i] = buf[(p * S + (lo >> 1)) * cap + (lo & 1) * room + (src - off[lo])];
        if (BITS) v[i] = make_key(__uint_as_float((uint32_t)(v[i] >> 32)), (uint32_t)v[i]);
      }
    }
    next += fresh;
    uint32_t t_hi = 0xffffffffu, t_lo = 0xffffffffu;  // the last key to keep
    if (m > pool) {
      // from the highest bit in which two keys differ
      const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)(v[0] >> 32));
      uint32_t diff = 0;
#pragma unroll
      for (int i = 0; i < E; ++i)
        if (i * 64 + lane < m) diff |= (uint32_t)(v[i] >> 32) ^ first;
      int bit = 31 - __clz((int)wave_or_u32(diff));
      uint32_t prefix = bit < 31 ? first >> (bit + 1) << (bit + 1) : 0;
      bool cut = false;  // exactly `pool` keys lie at or below prefix
      for (; bit >= 0 && !cut; --bit) {
        const uint32_t t = prefix | ((1u << bit) - 1u);
        int c = 0;
        if constexpr (BITS) {  // k_collect's keys: many waves, and groups past m are skipped
#pragma unroll
          for (int i = 0; i < E; ++i)
            if (64 * i < m)
              c += __popcll(__builtin_amdgcn_ballot_w64((uint32_t)(v[i] >> 32) <= t));
        } else {
          c = wave_count<true, E>(
              [&](int i) { return (uint32_t)(v[i] >> 32) <= t && i * 64 + lane < m; });
        }
        cut = c == pool;
        prefix = cut ? t : c < pool ? prefix | (1u << bit) : prefix;
      }
      t_hi = prefix;
      int below = 0, upto = 0;
#pragma unroll
      for (int i = 0; i < E; ++i)
        if (64 * i < m && !cut) {
          below += __popcll(__builtin_amdgcn_ballot_w64((uint32_t)(v[i] >> 32) < t_hi));
          upto += __popcll(__builtin_amdgcn_ballot_w64((uint32_t)(v[i] >> 32) <= t_hi));
        }
      if (upto > pool) {  // equal distances at the cut: the lower indices stay
        prefix = 0;
        for (int bit = 31; bit >= 0; --bit) {
          const uint32_t t = prefix | ((1u << bit) - 1u);
          int c = below;
#pragma unroll
          for (int i = 0; i < E; ++i)
            if (64 * i < m)
              c += __popcll(__builtin_amdgcn_ballot_w64((uint32_t)(v[i] >> 32) == t_hi &&
                                                        (uint32_t)v[i] <= t));
          if (c < pool) prefix |= 1u << bit;
        }
        t_lo = prefix;
      }
    }
    const uint64_t last = ((uint64_t)t_hi << 32) | t_lo;
    have = 0;
#pragma unroll
    for (int i = 0; i < E; ++i)
      if (64 * i < m) {
        const bool keep = i * 64 + lane < m && v[i] <= last;
        const uint64_t mask = __builtin_amdgcn_ballot_w64(keep);
        if (keep) kept[have + __popcll(mask & ((1ull << lane) - 1ull))] = v[i];
        have += __popcll(mask);
      }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } while (next < total);
  uint64_t s[PE];
#pragma unroll
  for (int i = 0; i < PE; ++i) s[i] = lane * PE + i < have ? kept[lane * PE + i] : ~0ull;
  wave_bitonic_sort<PE>(s);
  const int64_t q = list ? list[list_base + p] : p;
#pragma unroll
  for (int i = 0; i < PE; ++i)
    if (lane * PE + i < have) out[q * pool + lane * PE + i] = s[i];
  if (lane == 0) out_cnt[q] = have;
}

// Exact FP64 squared distance, terms added in feature order, no contraction: the
// same evaluation as the CPU oracle, so results agree bit for bit.
__device__ __forceinline__ double sqdist_exact(const float *__restrict__ q_lds,
                                               const float *__restrict__ r, int D) {
#pragma clang fp contract(off)
  double acc = 0.0;
  int t = 0;
  if ((reinterpret_cast<uintptr_t>(r) & 7) == 0) {
    // 8-byte rows: half the load instructions (each lane reads a different row), the
    // same terms in the same order
    const float2 *r2 = reinterpret_cast<const float2 *>(r);
    for (; t + 1 < D; t += 2) {
      const float2 rv = r2[t >> 1];
      double df = (double)q_lds[t] - (double)rv.x;
      double sq = df * df;
      acc = acc + sq;
      df = (double)q_lds[t + 1] - (double)rv.y;
      sq = df * df;
      acc = acc + sq;
    }
  }
  for (; t < D; ++t) {
    double df = (double)q_lds[t] - (double)r[t];
    double sq = df * df;
    acc = acc + sq;
  }
  return acc;
}

// sqdist_exact of one row per lane, for a wave: lane i < n has row j (any valid one elsewhere).
// A lane reading its own row touches 64 rows an instruction, 25 times over at D = 50, and 64
// rows a wave are more than L1 holds between two of them.  So the wave loads rows together,
// 128 bytes of eight rows an instruction (16 bytes a lane, on rows aligned to 4), through LDS,
// with the next 32 features in flight while these are added, in the same order.  36 floats a
// row: sixteen lanes' 16-byte reads meet no bank twice.
constexpr int kRankFeat = 32, kRankRow = kRankFeat + 4;
struct __attribute__((packed, aligned(4))) RankPiece {
  float x[4];
};
__device__ __forceinline__ double sqdist_rows(const float *q_lds, const float *__restrict__ R,
                                              int64_t ldr, int D, uint32_t j, int n,
                                              float *tile) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, sub = lane & 7, r8 = lane >> 3;
  const float *row[8];
#pragma unroll
  for (int u = 0; u < 8; ++u)
    row[u] = R + (int64_t)(uint32_t)__shfl((int)j, 8 * u + r8, kWave) * ldr;
  RankPiece w[8];
  auto load = [&](int t0) {
    const int f = t0 + 4 * sub;
    if (f + 4 <= D) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (8 * u < n) w[u] = *reinterpret_cast<const RankPiece *>(row[u] + f);
    } else if (f < D) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (8 * u < n) {
          w[u].x[0] = row[u][f];
          if (f + 1 < D) w[u].x[1] = row[u][f + 1];
          if (f + 2 < D) w[u].x[2] = row[u][f + 2];
        }
    }
  };
  load(0);
  double acc = 0.0;
  for (int t0 = 0; t0 < D; t0 += kRankFeat) {
    if (t0 + 4 * sub < D) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (8 * u < n)
          *reinterpret_cast<float4 *>(tile + (8 * u + r8) * kRankRow + 4 * sub) =
              make_float4(w[u].x[0], w[u].x[1], w[u].x[2], w[u].x[3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (t0 + kRankFeat < D) load(t0 + kRankFeat);
    const int here = min(kRankFeat, D - t0);
    const float *mine = tile + lane * kRankRow;
    auto add = [&](float a, float b) {
      const double df = (double)a - (double)b;
      const double sq = df * df;
      acc = acc + sq;
    };
    int t = 0;
#pragma unroll 4
    for (; t + 4 <= here; t += 4) {
      const float4 a = *reinterpret_cast<const float4 *>(q_lds + t0 + t);
      const float4 b = *reinterpret_cast<const float4 *>(mine + t);
      add(a.x, b.x);
      add(a.y, b.y);
      add(a.z, b.z);
      add(a.w, b.w);
    }
    for (; t < here; ++t) add(q_lds[t0 + t], mine[t]);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  return acc;
}

// One wave per query: merge the slices' pools to the global best `pool` by screened
// key, re-rank them exactly, take the best k (+1 with self repair).
// Consecutive queries share candidates and an L2: the grid is a multiple of the eight XCDs, which
// take workgroups in turn, and each XCD gets a contiguous eighth of the queries.
// Rows in turn through LDS from here on (us of the kernel with a row a lane / through LDS, D = 50,
// pool 64): 1 query 7.3 / 7.1 of 500,000 references and 5.4 / 6.2 of 20,000, 256 queries 8.1 /
// 7.8 and 6.4 / 7.4, 1000 9.2 / 9.2 and 8.6 / 8.5, 2000 13.4 / 12.8 and 11.9 / 10.9, 16,000
// 71 / 48 and 45 / 39.  Whole searches: 1,000,000 cells 3.61 -> 2.93 ms of rerank, 1,500,000
// with pools of 128 22.3 -> 13.8; 16 features at a time give 2.65 and 15.7.
constexpr int64_t kRankRowsFrom = 1024;
template <int PE, bool ROWS>  // pool elements per lane (pool <= 64 * PE), sqdist_rows
__global__ void __launch_bounds__(256) k_rerank(
    const float *__restrict__ Q, int64_t nq, int64_t ldq, const float *__restrict__ R,
    int64_t nr, int64_t ldr, int32_t D, const uint64_t *__restrict__ cand,
    const int32_t *__restrict__ cand_cnt, int pool, int S, int k, int64_t self_offset,
    const int64_t *__restrict__ self_idx,
    double err_coef, float r_norm_max, double margin, int64_t *__restrict__ idx_out,
    float *__restrict__ dist_out, int32_t *__restrict__ flags) {
  __shared__ __attribute__((aligned(16))) float qv[4][256], tile[ROWS ? 4 : 1][64 * kRankRow];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t block = (int64_t)(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  const int64_t q = block * 4 + w;
  if (q >= nq) return;
  float *ql = qv[w];
  for (int t = lane; t < D; t += 64) ql[t] = Q[q * ldq + t];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();

  // 1. merged pool: best `pool` keys over the S slices
  uint64_t v[PE];
  int total = 0;
  {
    const int c0 = cand_cnt[q * S];
    const uint64_t *p0 = cand + (q * S) * pool;
#pragma unroll
    for (int i = 0; i < PE; ++i) {
      const int e = lane * PE + i;
      v[i] = e < c0 ? p0[e] : ~0ull;
    }
    total = c0;
  }
  for (int s = 1; s < S; ++s) {
    const int cs = cand_cnt[q * S + s];
    const uint64_t *ps = cand + (q * S + s) * pool;
    uint64_t m[2 * PE];
#pragma unroll
    for (int i = 0; i < PE; ++i) m[i] = v[i];
    // second half of the 2*PE-per-lane array: the new slice
#pragma unroll
    for (int i = 0; i < PE; ++i) {
      const int e = lane * PE + i;
      m[PE + i] = e < cs ? ps[e] : ~0ull;
    }
    wave_bitonic_sort<2 * PE>(m);
    // the best `pool` now sit at elements 0..pool-1 = lanes 0..pool/(2PE)-1; move
    // them back to the PE-per-lane layout: element e lives at lane e/(2PE), slot e%(2PE)
#pragma unroll
    for (int i = 0; i < PE; ++i) {
      const int e = lane * PE + i;
      const int src = e / (2 * PE), slot = e % (2 * PE);
      uint64_t mine = 0;
      // every lane offers its slot `slot`... gather with a shuffle per slot value
#pragma unroll
      for (int sl = 0; sl < 2 * PE; ++sl) {
        uint32_t lo = __shfl((uint32_t)m[sl], src, kWave);
        uint32_t hi = __shfl((uint32_t)(m[sl] >> 32), src, kWave);
        if (sl == slot) mine = ((uint64_t)hi << 32) | lo;
      }
      v[i] = mine;
    }
    total += cs;
  }
  const int npool = total < pool ? total : pool;
  // screened key of the pool's last element: the bound on everything left out
  const uint64_t lastkey = wave_elem_u64<PE>(v, npool > 0 ? npool - 1 : 0);

  // 2. exact distances of the pool
  double qn = 0.0;  // ||q||^2 in FP64 (the certificate and the margin test)
  if (err_coef >= 0.0 || margin > 0.0)
    for (int t = 0; t < D; ++t) qn += (double)ql[t] * (double)ql[t];
  KeyIdx c[PE];
  double emax = 0.0;  // largest screening error |key + ||q||^2 - exact| over the pool
#pragma unroll
  for (int i = 0; i < PE; ++i) {
    const int e = lane * PE + i;
    const uint32_t j = (uint32_t)v[i];
    double dist = 0.0;
    if (ROWS && i < npool) {
      const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)j);
      dist = sqdist_rows(ql, R, ldr, D, e < npool ? j : first, (npool - i + PE - 1) / PE, tile[w]);
    }
    if (e < npool) {
      c[i].d = ROWS ? dist : sqdist_exact(ql, R + (int64_t)j * ldr, D);
      c[i].i = j;
      if (margin > 0.0)
        emax = fmax(emax, fabs((double)ord_float((uint32_t)(v[i] >> 32)) + qn - c[i].d));
    } else {
      c[i].d = INFINITY;
      c[i].i = 0xffffffffu;
    }
  }
  if (margin > 0.0) emax = wave_max_f64(emax);
  wave_bitonic_sort<PE>(c);

  const bool self = self_idx != nullptr || self_offset >= 0;
  const int kk = self ? k + 1 : k;
  // broadcast the first kk (<= 64*PE) sorted elements through LDS-free shuffles
  // element e is at lane e/PE, slot e%PE
  int32_t flag = 0;
  // certificate: every reference outside the pool has exact distance
  // >= lastkey + ||q||^2 - err; the k-th chosen one must be strictly below that.
  // References were left out whenever the index holds more rows than the merged pool
  // (each slice stores at most `pool` keys, so `total` cannot tell with one slice).
  if (err_coef >= 0.0) {
    bool certified = true;
    if (nr > (int64_t)npool && kk > 0) {
      const double rq = sqrt(qn);
      const double err =
          err_coef * ((double)r_norm_max * r_norm_max + 2.0 * rq * (double)r_norm_max + qn);
      const double bound = (double)ord_float((uint32_t)(lastkey >> 32)) + qn - err;
      // kk-th exact distance (element kk-1)
      const int e = (kk <= npool ? kk : npool) - 1;
      double dk = 0.0;
      {
        double mine = 0.0;
#pragma unroll
        for (int i = 0; i < PE; ++i)
          if (lane * PE + i == e) mine = c[i].d;
        dk = __shfl(mine, e / PE, kWave);
      }
      certified = dk < bound;
    }
    if (!certified) flag |= SH_FLAG_UNCERTIFIED;
  }
  // margin test of a low-precision screen: a reference left out of the pool has a
  // screened key >= lastkey, so a true neighbour was lost only if its screening error
  // reached gap = lastkey + ||q||^2 - d_kk.  The pool shows the errors the screen made
  // near this query; rows whose gap is under margin times the largest of them are
  // flagged for a wider second screen.
  if (margin > 0.0 && nr > (int64_t)npool && kk > 0) {
    const int e = (kk <= npool ? kk : npool) - 1;
    double mine = 0.0;
#pragma unroll
    for (int i = 0; i < PE; ++i)
      if (lane * PE + i == e) mine = c[i].d;
    const double dk = __shfl(mine, e / PE, kWave);
    const double gap = (double)ord_float((uint32_t)(lastkey >> 32)) + qn - dk;
    if (gap <= margin * emax) flag |= SH_FLAG_THIN;
  }
  // gather the top kk (index, distance) into lane-indexed registers: lane t <- elem t
  double dd[2];
  uint32_t ii[2];
#pragma unroll
  for (int rep = 0; rep < 2; ++rep) {
    const int e = lane + 64 * rep;
    const int src = (e < 64 * PE ? e : 0) / PE, slot = e % PE;
    double dm = INFINITY;
    uint32_t im = 0xffffffffu;
#pragma unroll
    for (int sl = 0; sl < PE; ++sl) {
      double t_d = __shfl(c[sl].d, src, kWave);
      uint32_t t_i = (uint32_t)__shfl((int)c[sl].i, src, kWave);
      if (sl == slot) {
        dm = t_d;
        im = t_i;
      }
    }
    if (e >= npool) {
      dm = INFINITY;
      im = 0xffffffffu;
    }
    dd[rep] = dm;
    ii[rep] = im;
  }
  // self repair (ann.py:31-52) on the kk = k+1 list
  int drop = -1;
  if (self) {
    const int64_t me = self_idx ? self_idx[q] : self_offset + q;
    int pos = -1;
    for (int e = 0; e < kk; ++e) {
      const uint32_t ie = (uint32_t)__shfl((int)ii[e / 64], e % 64, kWave);
      if ((int64_t)ie == me) {
        pos = e;
        break;
      }
    }
    if (pos < 0) {
      drop = kk - 1;
      flag |= SH_FLAG_SELF_MISSING;
    } else {
      drop = pos;
    }
    if (pos != 0) flag |= SH_FLAG_SELF_NOT_FIRST;
  }
  // output column col takes element col (col < drop) or col + 1 (col >= drop); the
  // element may sit in another lane: shuffle
#pragma unroll
  for (int rep = 0; rep < 2; ++rep) {
    const int col = lane + 64 * rep;
    const int e = (drop >= 0 && col >= drop) ? col + 1 : col;
    const int esrc = e < 128 ? e : 127;
    double d0 = __shfl(dd[0], esrc % 64, kWave), d1 = __shfl(dd[1], esrc % 64, kWave);
    uint32_t i0 = (uint32_t)__shfl((int)ii[0], esrc % 64, kWave);
    uint32_t i1 = (uint32_t)__shfl((int)ii[1], esrc % 64, kWave);
    const double de = esrc < 64 ? d0 : d1;
    const uint32_t ie = esrc < 64 ? i0 : i1;
    if (col < k) {
      idx_out[q * k + col] = ie == 0xffffffffu ? -1 : (int64_t)ie;
      dist_out[q * k + col] = (float)de;
    }
  }
  if (flags && lane == 0) flags[q] = flag;
}

// FP64 brute force over all references for selected query rows (rows the
// certificate rejected, or every row when used as the FP64 reference).  One wave per
// query; each lane keeps a sorted top-KK of the references it visits
// (lane, lane + 64, ...), then the wave sorts the 64 * KK survivors.
template <int KK>
__global__ void __launch_bounds__(256) k_exact(
    const float *__restrict__ Q, int64_t ldq, const int64_t *__restrict__ q_rows, int64_t n_sel,
    const float *__restrict__ R, int64_t nr, int64_t ldr, int32_t D, int k, int64_t self_offset,
    const int64_t *__restrict__ self_idx,
    int64_t *__restrict__ idx_out, float *__restrict__ dist_out, double *__restrict__ dist64_out,
    int32_t *__restrict__ flags) {
  __shared__ float qv[4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t sel = (int64_t)blockIdx.x * 4 + w;
  if (sel >= n_sel) return;
  const int64_t q = q_rows ? q_rows[sel] : sel;
  float *ql = qv[w];
  for (int t = lane; t < D; t += 64) ql[t] = Q[q * ldq + t];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  KeyIdx best[KK];
#pragma unroll
  for (int i = 0; i < KK; ++i) {
    best[i].d = INFINITY;
    best[i].i = 0xffffffffu;
  }
  for (int64_t j = lane; j < nr; j += 64) {
    KeyIdx x;
    x.d = sqdist_exact(ql, R + j * ldr, D);
    x.i = (uint32_t)j;
    if (less_ki(x, best[KK - 1])) {
#pragma unroll
      for (int p = KK - 1; p >= 0; --p) {
        const bool here = less_ki(x, best[p]);
        const bool prev = p > 0 && less_ki(x, best[p - 1]);
        if (here) best[p] = prev ? best[p - 1] : x;
      }
    }
  }
  wave_bitonic_sort<KK>(best);
  const bool self = self_idx != nullptr || self_offset >= 0;
  const int kk = self ? k + 1 : k;
  int drop = -1;
  int32_t flag = 0;
  if (self) {
    const int64_t me = self_idx ? self_idx[q] : self_offset + q;
    int pos = -1;
    for (int e = 0; e < kk; ++e) {
      uint32_t mine = 0;
#pragma unroll
      for (int i = 0; i < KK; ++i)
        if (lane * KK + i == e) mine = best[i].i;
      const uint32_t ie = (uint32_t)__shfl((int)mine, e / KK, kWave);
      if ((int64_t)ie == me) {
        pos = e;
        break;
      }
    }
    drop = pos < 0 ? kk - 1 : pos;
    if (pos < 0) flag |= SH_FLAG_SELF_MISSING;
    if (pos != 0) flag |= SH_FLAG_SELF_NOT_FIRST;
  }
  for (int col = 0; col < k; ++col) {
    const int e = (drop >= 0 && col >= drop) ? col + 1 : col;
    double md = 0.0;
    uint32_t mi = 0;
#pragma unroll
    for (int i = 0; i < KK; ++i)
      if (lane * KK + i == e) {
        md = best[i].d;
        mi = best[i].i;
      }
    const double de = __shfl(md, e / KK, kWave);
    const uint32_t ie = (uint32_t)__shfl((int)mi, e / KK, kWave);
    if (lane == 0) {
      idx_out[q * k + col] = ie == 0xffffffffu ? -1 : (int64_t)ie;
      dist_out[q * k + col] = (float)de;
      if (dist64_out) dist64_out[q * k + col] = de;
    }
  }
  // a row recomputed here after the re-rank's certificate failed keeps that flag
  if (flags && lane == 0) flags[q] = (flags[q] & SH_FLAG_UNCERTIFIED) | flag;
}


// fix_knn_query (ann.py:31-52) on a (k+1)-column table, one thread per row: drop the
// query's own column (column 0 in the common case), else the last column.
__global__ void k_fix_knn(const int64_t *__restrict__ idx_in, const float *__restrict__ dist_in,
                          const int64_t *__restrict__ ref_idx, int64_t n, int k1,
                          int64_t *__restrict__ idx_out, float *__restrict__ dist_out,
                          int32_t *__restrict__ flags) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t me = ref_idx[i];
  int pos = -1;
  for (int e = 0; e < k1; ++e)
    if (idx_in[i * k1 + e] == me) {
      pos = e;
      break;
    }
  int32_t flag = 0;
  if (pos != 0) flag |= SH_FLAG_SELF_NOT_FIRST;
  if (pos < 0) flag |= SH_FLAG_SELF_MISSING;
  const int drop = pos < 0 ? k1 - 1 : pos;
  for (int c = 0; c < k1 - 1; ++c) {
    const int e = c < drop ? c : c + 1;
    idx_out[i * (k1 - 1) + c] = idx_in[i * k1 + e];
    dist_out[i * (k1 - 1) + c] = dist_in[i * k1 + e];
  }
  if (flags) flags[i] = flag;
}

}  // namespace sh

using namespace sh;

extern "C" int sh_fix_knn_query(const int64_t *idx_in, const float *dist_in,
                                const int64_t *ref_idx, int64_t n, int32_t k1, int64_t *idx_out,
                                float *dist_out, int32_t *flags_out, sh_stream_t stream) {
  SH_ARG(n >= 0 && k1 >= 2, "sh_fix_knn_query: need n >= 0 and at least 2 columns");
  SH_ARG(idx_in && dist_in && ref_idx && idx_out && dist_out, "sh_fix_knn_query: NULL pointer");
  if (n == 0) return SH_OK;
  hipLaunchKernelGGL(k_fix_knn, dim3(cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, idx_in,
                     dist_in, ref_idx, n, k1, idx_out, dist_out, flags_out);
  SH_LAUNCH_CHECK("k_fix_knn");
  return SH_OK;
}

extern "C" int32_t sh_knn_pack_k(int dtype, int32_t D) { return pack_k(dtype, D); }
extern "C" int64_t sh_knn_pack_row_bytes(int dtype, int32_t D) { return pack_row_bytes(dtype, D); }

extern "C" int sh_knn_pack(const float *E, int64_t n, int32_t D, int64_t lde, int dtype, int role,
                           void *out, float *aux_out, sh_stream_t stream) {
  SH_ARG(n >= 0 && D > 0 && D <= 128 && lde >= D, "sh_knn_pack: bad sizes D=%d lde=%lld", D,
         (long long)lde);
  SH_ARG(role == 0 || role == 1, "sh_knn_pack: role must be 0 (reference) or 1 (query)");
  SH_ARG(E && out, "sh_knn_pack: NULL pointer");
  const int32_t K = pack_k(dtype, D);
  if (K < 0) {
    set_error("sh_knn_pack: unsupported dtype %d", dtype);
    return SH_EUNSUPPORTED;
  }
  if (n == 0) return SH_OK;
  // fewer rows a workgroup where the batch would leave the GPU idle
  const int rb = n >= 64 * 512 ? kPackRows : n >= 16 * 256 ? 16 : 4;
  const dim3 grid((uint32_t)cdiv(n, rb)), block(kPackThreads);
  const size_t lds = (size_t)rb * (D | 1) * sizeof(float);
#define SH_PACK(DT)                                                                             \
  hipLaunchKernelGGL(k_pack<DT>, grid, block, lds, (hipStream_t)stream, E, n, D, lde, role, K,  \
                     rb, (uint32_t *)out, aux_out)
  if (dtype == SH_F32)
    SH_PACK(SH_F32);
  else if (dtype == SH_BF16)
    SH_PACK(SH_BF16);
  else
    SH_PACK(SH_FP8);
#undef SH_PACK
  SH_LAUNCH_CHECK("k_pack");
  return SH_OK;
}

static int screen_cap(int pool) { return pool <= 64 ? 256 : pool <= 128 ? 512 : 1024; }

extern "C" size_t sh_knn_screen_workspace(int64_t nq, int32_t pool, int32_t n_slices) {
  return (size_t)nq * n_slices * screen_cap(pool) * sizeof(uint64_t);
}

// The operand type's launchers (all NULL for an unknown type).
static KnnOps knn_ops(int dtype) {
  return dtype == SH_BF16  ? knn_ops_bf16()
         : dtype == SH_FP8 ? knn_ops_fp8()
         : dtype == SH_F32 ? knn_ops_f32()
                           : KnnOps{};
}

extern "C" int sh_knn_screen(const void *qpack, int64_t nq, const void *rpack, int64_t nr,
                             int32_t D, int dtype, const float *q_aux, const float *r_aux,
                             int32_t pool, int32_t n_slices, const int64_t *seed_refs,
                             uint64_t *cand_keys, int32_t *cand_cnt, void *workspace,
                             size_t workspace_bytes, sh_stream_t stream) {
  (void)q_aux;
  (void)r_aux;
  SH_ARG(nq >= 0 && nr > 0 && D > 0, "sh_knn_screen: bad sizes nq=%lld nr=%lld D=%d",
         (long long)nq, (long long)nr, D);
  SH_ARG(nr < 0xffffffffll, "sh_knn_screen: more than 2^32-1 references");
  SH_ARG(pool >= 1 && pool <= 256, "sh_knn_screen: pool=%d outside [1, 256]", pool);
  SH_ARG(pool <= 128 || dtype == SH_FP8, "sh_knn_screen: pools above 128 are built for the FP8 "
         "screen only (pool=%d)", pool);
  SH_ARG(n_slices >= 1 && n_slices <= 4096, "sh_knn_screen: n_slices=%d", n_slices);
  SH_ARG(qpack && rpack && cand_keys && cand_cnt, "sh_knn_screen: NULL pointer");
  const size_t need = sh_knn_screen_workspace(nq, pool, n_slices);
  if (!workspace || workspace_bytes < need) {
    set_error("sh_knn_screen: workspace %zu < %zu bytes", workspace_bytes, need);
    return SH_EWORKSPACE;
  }
  if (nq == 0) return SH_OK;
  const int32_t K = pack_k(dtype, D);
  int64_t slice_len = align_up((size_t)cdiv(nr, n_slices), kSliceAlign);
  const int S = (int)cdiv(nr, slice_len);
  SH_ARG(S == n_slices, "sh_knn_screen: %d slices requested but %lld references give %d; use "
         "a slice count whose slices hold >= 128 references", n_slices, (long long)nr, S);
  SH_ARG(cdiv(nq, 128) <= 0x7fffffffll, "sh_knn_screen: too many queries");
  const KnnOps ops = knn_ops(dtype);
  ScreenArgs a = {};
  a.q = qpack, a.nq = nq, a.r = rpack, a.nr = nr, a.slice_len = slice_len;
  a.S = S, a.pool = pool, a.seeds = seed_refs;
  a.buf = (uint64_t *)workspace, a.out = cand_keys, a.out_cnt = cand_cnt;
  if (ops.screen && ops.screen(K, screen_cap(pool), a, (hipStream_t)stream)) {
    SH_LAUNCH_CHECK("k_screen");
    return SH_OK;
  }
  set_error("sh_knn_screen: dtype %d with packed K=%d not supported", dtype, K);
  return SH_EUNSUPPORTED;
}

// How sh_knn_pool cuts its work.
namespace sh {
struct PoolPlan {
  bool bounded;       // false: too few references for a threshold pass to pay
  bool collect;       // k_collect (and a second screen of what it lists), else k_screen
  int shift, rank;    // threshold pass: one sampled row of each 2^shift, rank of the minimum
  int64_t m;          // sampled rows
  int S1, per, slots; // slices, minima per lane half, slots per query
  int64_t len1;
  int64_t batch1;     // queries per threshold launch (bounds the slot workspace)
  int S3, cap;        // scan: slices, buffer keys per query and slice
  int64_t len3;
  int64_t batch3;     // queries per scan launch (bounds the candidate buffers)
  size_t off_slots, off_buf, off_cnt, off_fail, bytes;
};
constexpr int kCUs = 256;
constexpr size_t kSlotBytes = (size_t)1 << 30;
constexpr size_t kBufBytes = (size_t)4 << 30;
// k_collect's positions are bytes in 32 bits.  A lane half stops where its segment is full, but
// for keys of minus infinity, which pass any threshold: half of so many references (a lane
// half's) are 2^31 bytes of keys, beside less than 2^28 of segments.
constexpr int64_t kCollectRefs = (int64_t)1 << 29;
// Second screen: the first kAgain listed queries in kAgainSlices reference slices (a few
// failed queries must not wait for one workgroup's walk over all references), the rest
// kAgainBatch at a time in one slice.
constexpr int64_t kAgain = 4096;
constexpr int kAgainSlices = 16;
constexpr int64_t kAgainBatch = 1 << 18;

// Slices that fill `resident` workgroups: the first count from `lo` on whose last wave of
// workgroups leaves under 7% of the GPU idle, else the best one seen.
static int pick_slices(int64_t qblocks, int64_t resident, int lo, int hi) {
  int best = lo;
  double best_use = 0.0;
  for (int s = lo; s <= hi; ++s) {
    const int64_t wgs = qblocks * s;
    const double use = (double)wgs / (double)(cdiv(wgs, resident) * resident);
    if (use > best_use + 1e-9) {
      best_use = use;
      best = s;
    }
    if (best_use >= 0.93) break;
  }
  return best;
}

// Rank of the sampled minimum that becomes the threshold: of a pool the sample holds
// mean = pool / 2^shift on average (binomial, near Poisson), and exceeds
// mean + 4.75 sqrt(mean) + 5 with a chance of 1e-7 to 4e-7 for means from 1 to 64.
static int tau_rank(int pool, int shift) {
  const double mean = (double)pool / (1 << shift);
  return shift == 0 ? pool
                    : std::min(pool, (int)std::ceil(mean + 4.75 * std::sqrt(mean) + 5.0));
}

static PoolPlan pool_plan(int64_t nq, int64_t nr, int K, int dtype, int pool) {
  PoolPlan p = {};
  const KnnOps ops = knn_ops(dtype);
  const int64_t qb = std::max<int64_t>(1, cdiv(nq, 256));
  // A threshold pass pays where its sample can hold the pool, but not for a query or two of a few
  // hundred references, whose insertions take less than its two launches (whole calls, us,
  // without / with: one query, pool 64, 700 references 51 / 58, 1024 64 / 57; pool 20, 1500
  // 55 / 61, 2000 63 / 59; FP32, 512 136 / 125; two of 500, pool 64, 54 / 58; ten 127 / 58).
  p.bounded = nr >= 8 * (int64_t)pool &&
              (double)nq * (double)nr * std::sqrt((double)pool) * (dtype == SH_F32 ? 4 : 1) >= 8000.0;
  // Measured time of a pair in the scan's loop.
  const double c_pair = dtype == SH_F32    ? 0.75e-12 * K / 56
                        : dtype == SH_BF16 ? 0.1e-12 * K / 64
                                           : 0.055e-12 * K / 64;
  // Below some 5 us of scan the launches of the second screen cost what k_collect saves over
  // k_screen: whole calls take 61.7 us with k_screen and 63.5 with k_collect at 100 queries x
  // 100,000 references (BF16, D = 50), 88 and 81 at 1000 x 100,000, 155 and 135 at
  // 1000 x 500,000, 433 and 353 at 4000 x 500,000.
  p.collect = p.bounded && nr <= kCollectRefs && (double)nq * (double)nr * c_pair >= 5e-6;
  p.cap = screen_cap(pool);
  p.S1 = p.S3 = 1;
  p.len3 = align_up((size_t)nr, kSliceAlign);
  if (p.bounded) {
    // A sample of 1 / s of the rows costs nr * c_pair / s per query and leaves rank * s keys
    // (a tenth more for minima that share a slot) to insert.  Measured: a key costs 37 ps where a
    // tile of 32 references x 64 queries meets three of them and 80 ps where it meets one in two
    // tiles (the tile leaves the short path for it alone), twice that for FP8.  Self searches with
    // s = 1 / 2 / 4 / 8 / 16: a million cells 216 / 172 / 149 / 143 / 142 ms (16 is taken), 100,000
    // 2.92 / 2.64 / 2.43 / 2.41 / 2.55 (4), 19,001 in FP32 1.02 / 0.88 / 0.79 / 0.76 / 0.76 (8),
    // 300,000 in FP8 24.6 / 23.2 / 23.9 / 23.6 / 24.1 (4).
    double best = 0.0;
    for (int sh = 0; sh <= 4; ++sh) {
      if (sh > 0 && (nr >> sh) < 8 * (int64_t)pool) break;
      const int rank = p.collect ? tau_rank(pool, sh) : pool;
      const double keys = 1.1 * rank * (1 << sh);
      const double c_ins = (25e-12 + 75e-12 / (1.0 + keys * 2048.0 / (double)nr)) *
                           (dtype == SH_FP8 ? 2.0 : 1.0);
      const double cost = (double)nr * c_pair / (1 << sh) + keys * c_ins;
      if (sh == 0 || cost < best) {
        best = cost;
        p.shift = sh;
        p.rank = rank;
      }
    }
    p.m = nr >> p.shift;
    const int64_t res1 = (int64_t)ops.scan_resident(K) * kCUs;
    // at most 256 slices here and 512 below: one query's slots and segments are one wave's
    // work, and past that it takes longer than the slices save
    const int max1 = (int)std::min<int64_t>(256, cdiv(p.m, kSliceAlign));
    // slots enough that the rank-th smallest minimum is close to the rank-th smallest key
    const int min1 = (int)std::min<int64_t>(max1, cdiv(4 * (int64_t)p.rank, 16));
    const int want1 = (int)std::min<int64_t>(max1, cdiv(res1, qb));
    p.S1 = want1 > min1 ? want1 : pick_slices(qb, res1, min1, std::min(max1, min1 + 4));
    p.len1 = align_up((size_t)cdiv(p.m, p.S1), kSliceAlign);
    p.S1 = (int)cdiv(p.m, p.len1);
    p.per = 16 * p.S1 <= 512 ? 8 : 4 * p.S1 <= 512 ? 2 : 1;
    // more where the rank needs them, as many as k_tau takes (its rank is at most 256)
    while (p.per < 8 && p.S1 * 2 * p.per < 4 * p.rank)
      p.per = p.per == 1 ? 2 : 16 * p.S1 <= kTauSlots ? 8 : 4;
    p.slots = p.S1 * 2 * p.per;
    int64_t res3;
    if (p.collect) {
      res3 = (int64_t)ops.scan_resident(K) * kCUs;
      // a query's keys vary with the sample by 1 / sqrt(rank); all may come from one slice
      const double keys = 1.1 * p.rank * (1 << p.shift);
      p.cap = (int)align_up((size_t)(keys * (1.0 + 7.5 / std::sqrt((double)p.rank))) + 64, 128);
    } else {
      res3 = (int64_t)ops.screen_resident(K, p.cap) * kCUs;
    }
    // slices of at least 256 references, at most kBufBytes of candidate buffers
    const int64_t room = std::max<int64_t>(
        1, (int64_t)(kBufBytes / ((size_t)std::max<int64_t>(nq, 1) * p.cap * 8)));
    const int max3 = (int)std::min<int64_t>(std::min<int64_t>(p.collect ? 256 : 512, room),
                                            std::max<int64_t>(1, nr / 256));
    const int want3 = (int)cdiv(res3, qb);
    p.S3 = want3 >= max3 ? max3
                         : pick_slices(qb, res3, std::max(1, want3 - 1),
                                       std::min(max3, want3 + 6));
    p.len3 = align_up((size_t)cdiv(nr, p.S3), kSliceAlign);
    p.S3 = (int)cdiv(nr, p.len3);
  }
  p.batch1 = std::min<int64_t>(
      nq, std::max<int64_t>(256, (int64_t)(kSlotBytes / (std::max(p.slots, 1) * 4)) / 256 * 256));
  p.batch3 = nq;
  if (p.collect) {  // whole fills of the GPU a launch
    const int64_t most = (int64_t)(kBufBytes / ((size_t)p.S3 * p.cap * 8));
    const int64_t fill = (int64_t)ops.scan_resident(K) * kCUs * 256;
    p.batch3 = std::min(nq, most >= fill ? most / fill * fill
                                         : std::max<int64_t>(256, most / 256 * 256));
  }
  size_t o = align_up((size_t)nq * sizeof(float), 256);
  p.off_slots = o;
  if (p.bounded) o += align_up((size_t)p.batch1 * p.slots * sizeof(float), 256);
  p.off_buf = o;
  size_t keys = (size_t)p.batch3 * p.S3 * p.cap, segs = (size_t)p.batch3 * p.S3 * 2;
  if (p.collect) {
    const int cap2 = screen_cap(pool);
    const int64_t n1 = std::min(nq, kAgain), n2 = std::min(std::max<int64_t>(nq - kAgain, 0),
                                                           kAgainBatch);
    keys = std::max(keys, (size_t)std::max(n1 * kAgainSlices, n2) * cap2);
    segs = std::max(segs, (size_t)std::max(n1 * kAgainSlices, n2) * 2);
  }
  o += align_up(keys * sizeof(uint64_t), 256);
  p.off_cnt = o;
  if (p.collect || p.S3 > 1) o += align_up(segs * sizeof(int32_t), 256);
  p.off_fail = o;
  if (p.collect) o += 256 + align_up((size_t)nq * sizeof(int32_t), 256);
  p.bytes = o;
  return p;
}

// Whether the kernels that sh_knn_pool launches exist for this packed width.  pool_plan counts
// on it: it divides by the number of resident workgroups.
static bool pool_built(int dtype, int32_t D) {
  const KnnOps ops = knn_ops(dtype);
  const int32_t K = pack_k(dtype, D);
  return ops.bound && K > 0 && ops.scan_resident(K) > 0;
}

struct MergeArgs {
  const uint64_t *buf;
  const int32_t *seg_cnt;
  int64_t n;
  int S, cap, pool, need;
  const int32_t *list, *list_n;
  int32_t list_base;
  int32_t *fail, *fail_n;
  int32_t fail_base;
  uint64_t *out;
  int32_t *out_cnt;
};
template <bool BITS>
static void launch_merge(const MergeArgs &a, hipStream_t st) {
  const dim3 grid((uint32_t)cdiv(a.n, 4));
  const size_t lds = 4 * ((size_t)a.pool * sizeof(uint64_t) + 2 * (size_t)a.S * sizeof(int));
#define SH_MERGE(PE, E)                                                                        \
  hipLaunchKernelGGL((k_pool_merge<PE, E, BITS>), grid, dim3(256), lds, st, a.buf, a.seg_cnt, a.n,   \
                     a.S, a.cap, a.pool, a.need, a.list, a.list_n, a.list_base, a.fail,        \
                     a.fail_n, a.fail_base, a.out, a.out_cnt)
  if (a.pool <= 64)
    SH_MERGE(1, 8);
  else if (a.pool <= 128)
    SH_MERGE(2, 8);
  else
    SH_MERGE(4, 16);
#undef SH_MERGE
}
}  // namespace sh

extern "C" size_t sh_knn_pool_workspace(int64_t nq, int64_t nr, int32_t D, int dtype,
                                        int32_t pool) {
  if (nq <= 0 || nq > 0x7fffffffll || nr <= 0 || nr >= 0xffffffffll || D <= 0) return 0;
  if (pool < 1 || pool > (dtype == SH_FP8 ? 256 : 128) || !pool_built(dtype, D)) return 0;
  return pool_plan(nq, nr, pack_k(dtype, D), dtype, pool).bytes;
}

extern "C" int sh_knn_pool(const void *qpack, int64_t nq, const void *rpack, int64_t nr,
                           int32_t D, int dtype, int32_t pool, uint64_t *cand_keys,
                           int32_t *cand_cnt, void *workspace, size_t workspace_bytes,
                           sh_stream_t stream) {
  SH_ARG(nq >= 0 && nr > 0 && D > 0, "sh_knn_pool: bad sizes nq=%lld nr=%lld D=%d",
         (long long)nq, (long long)nr, D);
  SH_ARG(nr < 0xffffffffll, "sh_knn_pool: more than 2^32-1 references");
  SH_ARG(nq <= 0x7fffffffll, "sh_knn_pool: too many queries");
  SH_ARG(pool >= 1 && pool <= 256, "sh_knn_pool: pool=%d outside [1, 256]", pool);
  SH_ARG(pool <= 128 || dtype == SH_FP8, "sh_knn_pool: pools above 128 are built for the FP8 "
         "screen only (pool=%d)", pool);
  SH_ARG(qpack && rpack && cand_keys && cand_cnt, "sh_knn_pool: NULL pointer");
  const int32_t K = pack_k(dtype, D);
  const KnnOps ops = knn_ops(dtype);
  if (!pool_built(dtype, D)) {
    set_error("sh_knn_pool: dtype %d with packed K=%d not supported", dtype, K);
    return SH_EUNSUPPORTED;
  }
  if (nq == 0) return SH_OK;
  const PoolPlan p = pool_plan(nq, nr, K, dtype, pool);
  if (!workspace || workspace_bytes < p.bytes) {
    set_error("sh_knn_pool: workspace %zu < %zu bytes", workspace_bytes, p.bytes);
    return SH_EWORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  char *ws = (char *)workspace;
  float *tau0 = (float *)ws;
  float *slots = (float *)(ws + p.off_slots);
  uint64_t *buf = (uint64_t *)(ws + p.off_buf);
  int32_t *seg = (int32_t *)(ws + p.off_cnt);
  int32_t *fail_n = (int32_t *)(ws + p.off_fail), *fail = fail_n + 64;
  const int64_t qrow = pack_row_bytes(dtype, D);
  if (p.bounded) {
    for (int64_t q0 = 0; q0 < nq; q0 += p.batch1) {
      const int64_t nb = std::min(p.batch1, nq - q0);
      const BoundArgs b = {(const char *)qpack + q0 * qrow, nb,   rpack, p.m, p.shift, p.len1,
                           p.S1,                            p.per, slots};
      ops.bound(K, b, st);
      SH_LAUNCH_CHECK("k_bound");
      const dim3 grid((uint32_t)cdiv(nb, 4));
#define SH_TAU(EL)                                                                           \
  hipLaunchKernelGGL(k_tau<EL>, grid, dim3(256), 0, st, slots, nb, p.slots, p.rank, tau0 + q0, \
                     p.collect && q0 == 0 ? fail_n : nullptr)
      if (p.slots <= 64 * 2)
        SH_TAU(2);
      else if (p.slots <= 64 * 4)
        SH_TAU(4);
      else if (p.slots <= 64 * 8)
        SH_TAU(8);
      else
        SH_TAU(kTauSlots / 64);
#undef SH_TAU
      SH_LAUNCH_CHECK("k_tau");
    }
  }
  MergeArgs mg = {};
  mg.buf = buf, mg.seg_cnt = seg, mg.pool = pool;
  mg.need = (int)std::min<int64_t>(pool, nr);
  mg.out = cand_keys, mg.out_cnt = cand_cnt;
  ScreenArgs a = {};
  a.q = qpack, a.r = rpack, a.nr = nr, a.pool = pool, a.buf = buf;
  if (!p.collect) {
    a.nq = nq, a.slice_len = p.len3, a.S = p.S3;
    a.tau0 = p.bounded ? tau0 : nullptr;
    a.seg_cnt = p.S3 > 1 ? seg : nullptr;
    a.out = cand_keys, a.out_cnt = cand_cnt;
    if (!ops.screen(K, p.cap, a, st)) {
      set_error("sh_knn_pool: dtype %d with packed K=%d not supported", dtype, K);
      return SH_EUNSUPPORTED;
    }
    SH_LAUNCH_CHECK("k_screen");
    if (p.S3 > 1) {
      mg.n = nq, mg.S = p.S3, mg.cap = p.cap;
      launch_merge<false>(mg, st);
      SH_LAUNCH_CHECK("k_pool_merge");
    }
    return SH_OK;
  }
  for (int64_t q0 = 0; q0 < nq; q0 += p.batch3) {
    const int64_t nb = std::min(p.batch3, nq - q0);
    const CollectArgs c = {(const char *)qpack + q0 * qrow, nb,    rpack, nr, p.len3, p.S3,
                           tau0 + q0,                       p.cap, (uint2 *)buf, seg};
    ops.collect(K, c, st);
    SH_LAUNCH_CHECK("k_collect");
    MergeArgs m = mg;
    m.n = nb, m.S = p.S3, m.cap = p.cap;
    m.fail = fail, m.fail_n = fail_n, m.fail_base = (int32_t)q0;
    m.out = cand_keys + q0 * pool, m.out_cnt = cand_cnt + q0;
    launch_merge<true>(m, st);
    SH_LAUNCH_CHECK("k_pool_merge");
  }
  // the listed queries again, from an open threshold (their number stays on the device;
  // workgroups past it leave at once)
  for (int64_t base = 0; base < nq;) {
    const bool first = base == 0;
    const int64_t nb = std::min(nq - base, first ? kAgain : kAgainBatch);
    const int S = first ? (int)std::max<int64_t>(1, std::min<int64_t>(kAgainSlices, nr / 256)) : 1;
    a.nq = nb, a.slice_len = (int64_t)align_up((size_t)cdiv(nr, S), kSliceAlign);
    a.S = (int)cdiv(nr, a.slice_len);
    a.list = fail, a.list_n = fail_n, a.list_base = (int32_t)base;
    a.seg_cnt = seg;
    ops.screen(K, screen_cap(pool), a, st);
    SH_LAUNCH_CHECK("k_screen");
    MergeArgs m = mg;
    m.n = nb, m.S = a.S, m.cap = screen_cap(pool);
    m.list = fail, m.list_n = fail_n, m.list_base = (int32_t)base;
    launch_merge<false>(m, st);
    SH_LAUNCH_CHECK("k_pool_merge");
    base += nb;
  }
  return SH_OK;
}

extern "C" int sh_knn_rerank(const float *Q, int64_t nq, int64_t ldq, const float *R, int64_t nr,
                             int64_t ldr, int32_t D, const uint64_t *cand_keys,
                             const int32_t *cand_cnt, int32_t pool, int32_t n_slices, int32_t k,
                             int64_t self_offset, const int64_t *self_idx, double err_coef,
                             float r_norm_max, double margin,
                             int64_t *idx_out, float *dist_out, int32_t *flags_out,
                             sh_stream_t stream) {
  SH_ARG(nq >= 0 && nr > 0 && D > 0 && D <= 256, "sh_knn_rerank: bad sizes");
  SH_ARG(pool >= 1 && pool <= 256 && n_slices >= 1, "sh_knn_rerank: bad pool/slices");
  const int kk = k + ((self_offset >= 0 || self_idx) ? 1 : 0);
  SH_ARG(k >= 1 && kk <= pool && kk <= 127, "sh_knn_rerank: k=%d (+self) must be <= pool=%d", k,
         pool);
  SH_ARG(Q && R && cand_keys && cand_cnt && idx_out && dist_out, "sh_knn_rerank: NULL pointer");
  if (nq == 0) return SH_OK;
  const bool rows = nq >= kRankRowsFrom;
  auto kern = pool <= 64    ? (rows ? k_rerank<1, true> : k_rerank<1, false>)
              : pool <= 128 ? (rows ? k_rerank<2, true> : k_rerank<2, false>)
                            : (rows ? k_rerank<4, true> : k_rerank<4, false>);
  hipLaunchKernelGGL(kern, dim3((uint32_t)(8 * cdiv(cdiv(nq, 4), 8))), dim3(256), 0,
                     (hipStream_t)stream, Q, nq, ldq, R, nr, ldr, D, cand_keys, cand_cnt, pool,
                     n_slices, k, self_offset, self_idx, err_coef, r_norm_max, margin, idx_out,
                     dist_out, flags_out);
  SH_LAUNCH_CHECK("k_rerank");
  return SH_OK;
}

extern "C" int sh_knn_exact(const float *Q, int64_t nq, int64_t ldq, const int64_t *q_rows,
                            int64_t n_sel, const float *R, int64_t nr, int64_t ldr, int32_t D,
                            int32_t k, int64_t self_offset, const int64_t *self_idx,
                            int64_t *idx_out, float *dist_out,
                            double *dist64_out, int32_t *flags_out, sh_stream_t stream) {
  (void)nq;
  SH_ARG(n_sel >= 0 && nr > 0 && D > 0 && D <= 256, "sh_knn_exact: bad sizes");
  SH_ARG(nr < 0xffffffffll, "sh_knn_exact: more than 2^32-1 references");
  const int kk = k + ((self_offset >= 0 || self_idx) ? 1 : 0);
  SH_ARG(k >= 1 && kk <= 64, "sh_knn_exact: k=%d (+self) must be <= 64", k);
  SH_ARG(Q && R && idx_out && dist_out, "sh_knn_exact: NULL pointer");
  if (n_sel == 0) return SH_OK;
  dim3 grid(cdiv(n_sel, 4)), block(256);
  hipStream_t st = (hipStream_t)stream;
  if (kk <= 16)
    hipLaunchKernelGGL(k_exact<16>, grid, block, 0, st, Q, ldq, q_rows, n_sel, R, nr, ldr, D, k,
                       self_offset, self_idx, idx_out, dist_out, dist64_out, flags_out);
  else if (kk <= 32)
    hipLaunchKernelGGL(k_exact<32>, grid, block, 0, st, Q, ldq, q_rows, n_sel, R, nr, ldr, D, k,
                       self_offset, self_idx, idx_out, dist_out, dist64_out, flags_out);
  else
    hipLaunchKernelGGL(k_exact<64>, grid, block, 0, st, Q, ldq, q_rows, n_sel, R, nr, ldr, D, k,
                       self_offset, self_idx, idx_out, dist_out, dist64_out, flags_out);
  SH_LAUNCH_CHECK("k_exact");
  return SH_OK;
}
