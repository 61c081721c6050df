// The kNN screen and threshold kernels (templates) and their launch interface.
//
// One translation unit per operand type instantiates them (sh_knn_{bf16,fp8,f32}.hip);
// sh_knn.hip holds everything that does not depend on the operand type.
//
// Screen: the MFMA computes s(q, r) = ||r||^2 - 2 q.r directly: reference rows are
// packed as [r, ||r||^2 (split over 1 or 3 slots), 0...] and query rows as
// [-2q, 1, ..., 0...], so one K-padded dot product gives the ranking key
// (||q||^2 is the same for every reference of a query and is left out).
//   A operand = 32 references, B operand = 32 queries, D = 32 x 32 FP32 tile: lane l
//   holds query l%32 and 16 references 8*(v/4) + 4*(l/32) + v%4.
// The K axis is split between the two lane halves: half h supplies elements
// [h*K/2, (h+1)*K/2) of its row, for both operands, so each lane streams one
// contiguous half-row (the MFMA pairs A and B by the same (half, element) slot,
// so any such split gives the same dot product).
//
// Selection: per (query, reference slice) a candidate buffer of CAP (key, index)
// pairs in global memory and a threshold tau = the pool-th best key so far.  A
// 32 x 32 tile is filtered with a 16-value min tree and one compare per query;
// only tiles with a hit (rare once tau has settled) take the insertion path.  When
// a buffer nears CAP the owning wave sorts it (bitonic across the wave) and keeps
// the best `pool`.  References come in index order and the lower index wins a tie, so from
// then on tau excludes the pool-th key itself: a query with many equal references would
// otherwise insert them all.  Each wave owns its queries, so no cross-wave synchronisation.
// Optionally each query block first screens a set of seed reference rows (for self
// queries in locality order: the block's own rows) and starts tau at their pool-th key.
#pragma once
#include <float.h>

#include <type_traits>

#include "sh_common.h"
#include "sh_wave_sort.h"

namespace sh {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------------
// Screen kernel.
struct OpF32 {
  typedef float Frag;
  static constexpr int EPL = 1;  // elements per lane per MFMA
  static constexpr int ESZ = 4;
  static constexpr bool kScaled = false;
  static __device__ __forceinline__ floatx16 mma(Frag a, Frag b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
};
struct OpBF16 {
  typedef bf16x8 Frag;
  static constexpr int EPL = 8;
  static constexpr int ESZ = 2;
  static constexpr bool kScaled = false;
  static __device__ __forceinline__ floatx16 mma(Frag a, Frag b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
// FP8 E4M3 with per-row E8M0 scales (MX-style, one scale per lane's 32-element block):
// the norms enter through the accumulator, read from each row's 16-byte trailer.
typedef int intx8 __attribute__((ext_vector_type(8)));
struct OpFP8 {
  typedef intx8 Frag;
  static constexpr int EPL = 32;
  static constexpr int ESZ = 1;
  static constexpr bool kScaled = true;
  static __device__ __forceinline__ floatx16 mma_s(Frag a, Frag b, floatx16 c, int sa, int sb) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, sa, 0, sb);
  }
  static __device__ __forceinline__ floatx16 mma(Frag a, Frag b, floatx16 c) {
    return mma_s(a, b, c, 127, 127);
  }
};


constexpr int kSliceAlign = 128;       // reference slices start on this multiple
constexpr float kOpen = FLT_MAX;       // threshold of a pool that is not full yet

// QG: 32-query groups per wave; MINB: resident workgroups per CU the kernel is compiled
// for (its register budget).  Two groups at three workgroups per CU measured faster than
// four groups at two (BF16 K=64, 1M x 1M: 215 ms against 231 ms) and than one group at
// four (176 ms against 184 ms).
template <class Op, int K>
struct ScreenShape {
  static constexpr int QG = 2;
  static constexpr int QPB = 4 * 32 * QG;  // queries per workgroup
  static constexpr int MINB = 3;
};
// Register budget of one instantiation: three workgroups per CU (168 VGPRs) unless the
// query fragments or the compaction sort need more -- the FP8 screen at K >= 128 and the
// 1024-key buffers -- which then run two per CU instead of spilling to scratch.  The BF16
// screen at K <= 64 with 256-key buffers runs four per CU (128 VGPRs; its spills fall
// outside the tile loop): 166.6 against 174.6 ms at 1M x 1M, alternated runs on one GPU.
// The FP8 screen at K = 128 with 512-key buffers needs 165 VGPRs with the late index add
// (append_quad) and so runs three per CU instead of two.
template <class Op, int K, int CAP>
constexpr bool screen_late() {
  return (std::is_same<Op, OpBF16>::value && K <= 64 && CAP <= 256) ||
         (std::is_same<Op, OpFP8>::value && K > 64 && K <= 128 && CAP == 512);
}
template <class Op, int K, int CAP>
constexpr int screen_minb() {
  if constexpr (std::is_same<Op, OpBF16>::value && K <= 64 && CAP <= 256) return 4;
  if constexpr (std::is_same<Op, OpFP8>::value && K > 64 && K <= 128 && CAP == 512) return 3;
  return (Op::kScaled && K >= 128) || CAP >= 1024 ? 2 : ScreenShape<Op, K>::MINB;
}

// Candidate buffer of one (query, slice): CAP keys in two halves of CAP / 2, one per lane
// half (lanes n and n + 32 both serve query n); each lane appends to its own half with a
// register counter, so inserting needs no atomics.  Compaction (the whole wave, for one
// query) sorts both halves' c0 + c1 keys, keeps the best `pool` split between the two
// halves (or writes them to `out`), and returns the new threshold: the pool-th key once
// the query has seen `pool` candidates, else kOpen.
template <int CAP>
__device__ __forceinline__ int compact_pair(uint64_t *base, int c0, int c1, int pool,
                                            uint64_t *out, int32_t *out_cnt, float &tau_new) {
  constexpr int E = CAP / 64;
  constexpr int HALF = CAP / 2;
  const int lane = threadIdx.x & 63;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  uint64_t v[E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int e = lane * E + i;
    v[i] = e < c0 ? base[e] : (e - c0 < c1 ? base[HALF + (e - c0)] : ~0ull);
  }
  wave_bitonic_sort<E>(v);
  const int total = c0 + c1;
  const int keep = total < pool ? total : pool;
  const int k0 = (keep + 1) / 2;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int e = lane * E + i;
    if (e < keep) {
      if (out)
        out[e] = v[i];
      else
        base[e < k0 ? e : HALF + (e - k0)] = v[i];
    }
  }
  const uint64_t kp = wave_elem_u64<E>(v, pool - 1);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  if (out_cnt && lane == 0) *out_cnt = keep;
  tau_new = total >= pool ? ord_float((uint32_t)(kp >> 32)) : kOpen;
  return keep;
}

// True when the predicate holds on any lane of the wave (one ballot, no lane shuffles).
__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

// Appends this lane's values of one 4-reference quad that pass tau to its buffer half.
// Queries past the batch end carry tau = -inf, so nothing of theirs passes.
// LATE: the reference index is added inside the store (an asm statement the compiler
// cannot hoist).  Hoisted, a tile that takes this path computes all 16 indices and keeps
// them in registers, which the four-workgroups-per-CU budget cannot spare; at three per CU
// the hoisted form is faster.
template <int V, bool LATE>
__device__ __forceinline__ void append_one(const floatx16 &acc, float tau, uint32_t ref0,
                                           uint64_t *half, int &cnt) {
  constexpr int kOff = 8 * (V >> 2) + (V & 3);  // the value's reference within the tile
  if (acc[V] <= tau) {
    uint32_t ref;
    if constexpr (LATE)
      asm volatile("v_add_u32 %0, %1, %2" : "=v"(ref) : "i"(kOff), "v"(ref0));
    else
      ref = ref0 + (uint32_t)kOff;
    half[cnt] = make_key(acc[V], ref);
    ++cnt;
  }
}

template <int V0, bool LATE>
__device__ __forceinline__ void append_quad(const floatx16 &acc, float tau, uint32_t ref0,
                                            uint64_t *half, int &cnt) {
  append_one<V0, LATE>(acc, tau, ref0, half, cnt);
  append_one<V0 + 1, LATE>(acc, tau, ref0, half, cnt);
  append_one<V0 + 2, LATE>(acc, tau, ref0, half, cnt);
  append_one<V0 + 3, LATE>(acc, tau, ref0, half, cnt);
}

template <class Op, int K, int CAP>
__global__ void __launch_bounds__(256, (screen_minb<Op, K, CAP>())) k_screen(
    const typename Op::Frag *__restrict__ Qp_, int64_t nq, const unsigned char *__restrict__ Rp,
    int64_t nr, int64_t slice_len, int S, int pool, const int64_t *__restrict__ seeds,
    const float *__restrict__ tau0, const int32_t *__restrict__ list,
    const int32_t *__restrict__ list_n, int32_t list_base, uint64_t *__restrict__ buf,
    int32_t *__restrict__ seg_cnt, uint64_t *__restrict__ out, int32_t *__restrict__ out_cnt) {
  typedef typename Op::Frag Frag;
  constexpr int QG = ScreenShape<Op, K>::QG;
  constexpr bool kLate = screen_late<Op, K, CAP>();  // see append_quad
  constexpr int QPW = 32 * QG;                // queries per wave
  constexpr int QPB = ScreenShape<Op, K>::QPB;
  constexpr int HALFC = CAP / 2;              // keys per buffer half
  constexpr int HALF = K / 2;                 // elements per lane half
  constexpr int NS = HALF / Op::EPL;          // MFMA steps per tile
  constexpr int GROWB = K * Op::ESZ + (Op::kScaled ? 16 : 0);  // packed row bytes in HBM
  constexpr int ROWB = K * Op::ESZ + 16;      // LDS row bytes (pad or FP8 trailer)
  constexpr int CHUNKS = GROWB / 16;          // 16-byte chunks per packed row
  // references per LDS stage: as many as two stage buffers fit in 48 KiB
  constexpr int RT = (2 * 128 * ROWB <= 49152) ? 128 : (2 * 64 * ROWB <= 49152) ? 64 : 32;
  // stage buffers are filled by global_load_lds_dwordx4: each wave instruction writes
  // 64 consecutive 16-byte chunks (1 KiB), so a buffer is a whole number of KiB
  constexpr int CPR = ROWB / 16;                      // chunks per padded LDS row
  constexpr int NINSTR = (RT * CPR + 63) / 64;        // wave instructions per stage
  constexpr int BUFB = NINSTR * 1024;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_r[2][BUFB];

  const unsigned char *Qp = reinterpret_cast<const unsigned char *>(Qp_);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, n = lane & 31;
  const int slice = blockIdx.y;
  const int64_t r_begin = (int64_t)slice * slice_len;
  const int64_t r_end = min(nr, r_begin + slice_len);
  const int qw0 = w * QPW;  // wave's first local query
  const int64_t qb0 = (int64_t)blockIdx.x * QPB;
  // list mode: query position p stands for packed row list[list_base + p], and the number
  // of listed queries is known on the device only
  if (list) {
    nq = min(nq, (int64_t)*list_n - list_base);
    if (qb0 >= nq) return;
  }

  Frag bq[QG][NS];
  float tau[QG];
  bool qvalid[QG];
  int qscale[QG];
  int cnt[QG];
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const int64_t q = qb0 + qw0 + g * 32 + n;
    qvalid[g] = q < nq;
    // a query past the batch end never passes
    tau[g] = qvalid[g] ? (tau0 ? tau0[q] : kOpen) : -INFINITY;
    cnt[g] = 0;
    qscale[g] = 127;
    const int64_t row = qvalid[g] && list ? list[list_base + q] : q;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      bq[g][s] = qvalid[g] ? *reinterpret_cast<const Frag *>(
                                 Qp + row * GROWB + (h * HALF + s * Op::EPL) * Op::ESZ)
                           : Frag{};
    if (Op::kScaled && qvalid[g])
      qscale[g] = *reinterpret_cast<const int32_t *>(Qp + row * GROWB + K * Op::ESZ + 4);
  }

  // double buffering: stage t+1 streams into the other buffer (LDS DMA) while stage t
  // computes.  Chunk ci of a stage lands at byte 16*ci: row ci / CPR, column chunk
  // ci % CPR; the padding chunk of each row and rows past the slice re-read a valid
  // address (their values are never used).
  // Byte offset of this lane's chunk within a stage for each of its wave's instructions
  // (instruction j = w + 4 i fills LDS bytes [1024 j, 1024 j + 1024)); the padding chunk
  // of a row re-reads the row's first chunk (its value is never used).
  constexpr int JPW = (NINSTR + 3) / 4;  // instructions per wave per stage (at most)
  // rows the chunk layout touches per stage (can exceed RT by one when RT * CPR is not a
  // multiple of 64)
  constexpr int RROWS = (64 * NINSTR + CPR - 1) / CPR;
  uint32_t choff[JPW];
  int chrow[JPW];
#pragma unroll
  for (int i = 0; i < JPW; ++i) {
    const int ci = 64 * (w + 4 * i) + lane;
    const int rr = ci / CPR, c = ci % CPR;
    chrow[i] = rr;
    choff[i] = (uint32_t)(rr * GROWB + (c < CHUNKS ? c : 0) * 16);
  }
#define SH_SCREEN_FETCH(T0, B)                                                           \
  {                                                                                      \
    const unsigned char *stage = Rp + (T0) * GROWB;                                     \
    const bool whole = (T0) + RROWS <= r_end; /* uniform: no row past the slice */       \
    _Pragma("unroll") for (int i = 0; i < JPW; ++i) {                                    \
      const int j = w + 4 * i;                                                           \
      if (j < NINSTR) {                                                                  \
        const unsigned char *src;                                                        \
        if (whole) {                                                                     \
          src = stage + choff[i];                                                        \
        } else { /* rows past the slice re-read its last row */                          \
          const int64_t last = r_end - 1 - (T0);                                         \
          const int64_t over = chrow[i] > last ? (int64_t)chrow[i] - last : 0;           \
          src = stage + choff[i] - over * GROWB;                                         \
        }                                                                                \
        __builtin_amdgcn_global_load_lds(                                                \
            (const void *)src,                                                           \
            (__attribute__((address_space(3))) void *)(&lds_r[(B)][1024 * j]), 16, 0, 0); \
      }                                                                                  \
    }                                                                                    \
  }

  // Seeding: before the scan, every query of the workgroup screens the workgroup's QPB
  // seed references (seeds[qb0 .. qb0 + QPB), distinct rows of the reference set, e.g.
  // the block's own rows when queries are the references in locality order) and starts
  // from the pool-th smallest of those keys instead of an open threshold.  The seeds are
  // references of the slice, screened by the same MFMA arithmetic, so at least `pool`
  // references have a key at or below that threshold and the kept pool is the same; the
  // scan only skips candidates that could not have stayed.  (A 2^-16 relative margin
  // keeps this true even if a key were rounded differently in another tile position.)
  static_assert(QPB % 64 == 0 && QPB <= 256, "at most one seed slot per thread");
  static_assert(QPB % RT == 0 && (QPB / 32) * 16 <= HALFC, "seed stages must fit the buffer");
  if (seeds != nullptr && r_begin < r_end) {
    __shared__ uint32_t seed_row[QPB];
    __shared__ uint32_t seed_bad[QPB / 32];  // bit s of word i: slot 32 i + s has no seed
    if (threadIdx.x < QPB) {  // whole waves
      const int64_t q = qb0 + threadIdx.x;
      const int64_t r = q < nq ? seeds[q] : -1;
      const bool ok = r >= r_begin && r < r_end;
      seed_row[threadIdx.x] = (uint32_t)(ok ? r : r_begin);
      const uint64_t bad = __ballot(!ok);
      if (lane == 0) {
        seed_bad[2 * w] = (uint32_t)bad;
        seed_bad[2 * w + 1] = (uint32_t)(bad >> 32);
      }
    }
    __syncthreads();
    for (int s0 = 0; s0 < QPB; s0 += RT) {
      // gather the stage's seed rows: LDS row rr holds seed slot s0 + rr (rows the chunk
      // layout touches past the stage re-read a valid row; they are never used)
#pragma unroll
      for (int i = 0; i < JPW; ++i) {
        const int j = w + 4 * i;
        if (j < NINSTR) {
          const int slot = s0 + chrow[i];
          const uint32_t row = seed_row[slot < QPB ? slot : 0];
          const unsigned char *src =
              Rp + (int64_t)row * GROWB + (choff[i] - (uint32_t)(chrow[i] * GROWB));
          __builtin_amdgcn_global_load_lds(
              (const void *)src, (__attribute__((address_space(3))) void *)(&lds_r[0][1024 * j]),
              16, 0, 0);
        }
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
#pragma unroll
      for (int sub = 0; sub < RT / 32; ++sub) {
        floatx16 acc[QG];
        if constexpr (Op::kScaled) {
          floatx16 nrm;
#pragma unroll
          for (int v = 0; v < 16; ++v)
            nrm[v] = *reinterpret_cast<const float *>(
                &lds_r[0][(sub * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * ROWB + K * Op::ESZ]);
#pragma unroll
          for (int g = 0; g < QG; ++g) acc[g] = nrm;
        } else {
#pragma unroll
          for (int g = 0; g < QG; ++g)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[g][v] = 0.f;
        }
        const unsigned char *arow = &lds_r[0][(sub * 32 + n) * ROWB + h * HALF * Op::ESZ];
        int ascale = 127;
        if constexpr (Op::kScaled)
          ascale = *reinterpret_cast<const int32_t *>(
              &lds_r[0][(sub * 32 + n) * ROWB + K * Op::ESZ + 4]);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          Frag a = *reinterpret_cast<const Frag *>(arow + s * Op::EPL * Op::ESZ);
#pragma unroll
          for (int g = 0; g < QG; ++g) {
            if constexpr (Op::kScaled)
              acc[g] = Op::mma_s(a, bq[g][s], acc[g], ascale, qscale[g]);
            else
              acc[g] = Op::mma(a, bq[g][s], acc[g]);
          }
        }
        const uint32_t badw = seed_bad[(s0 >> 5) + sub];
#pragma unroll
        for (int g = 0; g < QG; ++g) {
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if ((badw >> (8 * (v >> 2) + 4 * h + (v & 3))) & 1u) acc[g][v] = INFINITY;
          const int64_t q = qb0 + qw0 + g * 32 + n;
          uint64_t *half = buf + ((qvalid[g] ? q : 0) * S + slice) * CAP + h * HALFC;
          append_quad<0, kLate>(acc[g], tau[g], 0u, half, cnt[g]);
          append_quad<4, kLate>(acc[g], tau[g], 0u, half, cnt[g]);
          append_quad<8, kLate>(acc[g], tau[g], 0u, half, cnt[g]);
          append_quad<12, kLate>(acc[g], tau[g], 0u, half, cnt[g]);
        }
      }
      __syncthreads();  // the next stage overwrites the buffer
    }
    // each query's threshold: the pool-th smallest seed key (open below `pool` seeds);
    // the seed keys themselves are dropped, the scan meets those references again
#pragma unroll
    for (int g = 0; g < QG; ++g) {
      for (int src = 0; src < 32; ++src) {
        const int64_t q = qb0 + qw0 + g * 32 + src;
        if (q >= nq) break;
        const int c0 = __builtin_amdgcn_readlane(cnt[g], src);
        const int c1 = __builtin_amdgcn_readlane(cnt[g], src + 32);
        float tnew;
        compact_pair<CAP>(buf + (q * S + slice) * CAP, c0, c1, pool, nullptr, nullptr, tnew);
        if (n == src)
          tau[g] = tnew < kOpen ? fminf(tnew + fabsf(tnew) * 0x1p-16f, kOpen) : kOpen;
      }
      cnt[g] = 0;
    }
  }

  const bool live = qb0 + qw0 < nq;  // a wave without queries only helps to stage
  int b = 0;
  if (r_begin < r_end) {
    SH_SCREEN_FETCH(r_begin, 0)
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int64_t t0 = r_begin; t0 < r_end; t0 += RT) {
    const int64_t tn = t0 + RT;
    if (tn < r_end) {
      SH_SCREEN_FETCH(tn, b ^ 1)
    }
#pragma unroll
    for (int sub = 0; sub < RT / 32; ++sub) {
      const int64_t rb = t0 + sub * 32;
      if (rb >= r_end || !live) continue;
      floatx16 acc[QG];
      if constexpr (Op::kScaled) {
        // accumulator starts at ||r||^2 of each of the lane's 16 references
        floatx16 nrm;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          nrm[v] = *reinterpret_cast<const float *>(
              &lds_r[b][(sub * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * ROWB + K * Op::ESZ]);
#pragma unroll
        for (int g = 0; g < QG; ++g) acc[g] = nrm;
      } else {
#pragma unroll
        for (int g = 0; g < QG; ++g)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[g][v] = 0.f;
      }
      const unsigned char *arow = &lds_r[b][(sub * 32 + n) * ROWB + h * HALF * Op::ESZ];
      // LLVM's small-GEMM interleave of the fragment LDS reads with the MFMAs: 175.1 ->
      // 172.3 ms for the 1M BF16 screen, alternated runs on one GPU
      __builtin_amdgcn_iglp_opt(0);
      int ascale = 127;
      if constexpr (Op::kScaled)
        ascale = *reinterpret_cast<const int32_t *>(&lds_r[b][(sub * 32 + n) * ROWB + K * Op::ESZ + 4]);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        Frag a = *reinterpret_cast<const Frag *>(arow + s * Op::EPL * Op::ESZ);
#pragma unroll
        for (int g = 0; g < QG; ++g) {
          if constexpr (Op::kScaled)
            acc[g] = Op::mma_s(a, bq[g][s], acc[g], ascale, qscale[g]);
          else
            acc[g] = Op::mma(a, bq[g][s], acc[g]);
        }
      }
      if (rb + 32 > r_end) {  // references past the slice end never pass
#pragma unroll
        for (int g = 0; g < QG; ++g)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int64_t ref = rb + 8 * (v >> 2) + 4 * h + (v & 3);
            if (ref >= r_end) acc[g][v] = INFINITY;
          }
      }
      // quad minima, then the tile minimum, per query group
      float m4[QG][4];
      bool hit[QG];
      bool any_hit = false;
#pragma unroll
      for (int g = 0; g < QG; ++g) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          m4[g][j] = fminf(fminf(acc[g][4 * j], acc[g][4 * j + 1]),
                           fminf(acc[g][4 * j + 2], acc[g][4 * j + 3]));
        const float m = fminf(fminf(m4[g][0], m4[g][1]), fminf(m4[g][2], m4[g][3]));
        hit[g] = m <= tau[g];
        any_hit |= hit[g];
      }
      if (wave_any(any_hit)) {
        // lane's first reference of the tile (quads add 8 * (v / 4) + v % 4)
        const uint32_t ref0 = (uint32_t)(rb + 4 * h);
#pragma unroll
        for (int g = 0; g < QG; ++g) {
          if (!wave_any(hit[g])) continue;
          const int64_t q = qb0 + qw0 + g * 32 + n;
          uint64_t *half = buf + ((qvalid[g] ? q : 0) * S + slice) * CAP + h * HALFC;
          if (wave_any(m4[g][0] <= tau[g]))
            append_quad<0, kLate>(acc[g], tau[g], ref0, half, cnt[g]);
          if (wave_any(m4[g][1] <= tau[g]))
            append_quad<4, kLate>(acc[g], tau[g], ref0, half, cnt[g]);
          if (wave_any(m4[g][2] <= tau[g]))
            append_quad<8, kLate>(acc[g], tau[g], ref0, half, cnt[g]);
          if (wave_any(m4[g][3] <= tau[g]))
            append_quad<12, kLate>(acc[g], tau[g], ref0, half, cnt[g]);
          // compact every query of the group one of whose halves cannot take a tile
          const uint64_t mk = __ballot(cnt[g] > HALFC - 16);
          uint32_t mq = (uint32_t)(mk | (mk >> 32));
          while (mq) {
            const int src = __ffs(mq) - 1;
            mq &= mq - 1;
            const int c0 = __builtin_amdgcn_readlane(cnt[g], src);
            const int c1 = __builtin_amdgcn_readlane(cnt[g], src + 32);
            const int64_t qs = qb0 + qw0 + g * 32 + src;
            float tnew;
            const int keep = compact_pair<CAP>(buf + (qs * S + slice) * CAP, c0, c1, pool,
                                               nullptr, nullptr, tnew);
            if (n == src) {
              cnt[g] = h == 0 ? (keep + 1) / 2 : keep - (keep + 1) / 2;
              // what comes now has a higher index, so of equal keys none can enter any more
              if (tnew < kOpen) tau[g] = fminf(tau[g], ord_float(float_ord(tnew) - 1));
            }
          }
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // the next stage's DMA has landed
    __syncthreads();
    b ^= 1;
  }
#undef SH_SCREEN_FETCH
  if (seg_cnt) {  // the keys stay in the buffer halves for k_pool_merge
#pragma unroll
    for (int g = 0; g < QG; ++g) {
      const int64_t q = qb0 + qw0 + g * 32 + n;
      if (qvalid[g]) seg_cnt[(q * S + slice) * 2 + h] = cnt[g];
    }
    return;
  }
  // final: sort each query's buffer and emit its best `pool`
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    for (int src = 0; src < 32; ++src) {
      const int64_t q = qb0 + qw0 + g * 32 + src;
      if (q >= nq) break;
      const int c0 = __builtin_amdgcn_readlane(cnt[g], src);
      const int c1 = __builtin_amdgcn_readlane(cnt[g], src + 32);
      float tnew;
      compact_pair<CAP>(buf + (q * S + slice) * CAP, c0, c1, pool, out + (q * S + slice) * pool,
                        out_cnt + q * S + slice, tnew);
    }
  }
}

// ---------------------------------------------------------------------------------
// Threshold pass: an upper bound of every query's pool-th smallest key, before the scan.
//
// The screen's cost beyond its MFMA loop is the insertions: a pool that starts open takes
// in pool * ln(references / pool) keys per query and slice on the way to its final
// threshold.  This pass runs the same MFMA tiles over a sample of the references (one row,
// at a hashed place, of each 2^shift consecutive ones) with no insertion path at all: each
// lane keeps the minimum of every accumulator register over its tiles.  A query's slot
// minima are keys of distinct references, so the pool-th smallest of them has at least
// `pool` references at or below it, and a scan that starts from it keeps the same pool.
// With 2^shift the scan meets about pool * 2^shift keys under that threshold.  Where the
// scan can screen a query again, a smaller rank is taken: the sample holds pool / 2^shift of
// the pool on average, and a rank that it exceeds with a chance of about 1e-7 leaves far
// fewer keys to insert (tau_rank in sh_knn.hip).
//
// slot_min[q][slice][2 * per]: a lane half keeps 8 minima (each of two accumulator
// registers, one v_min3 a pair), folded to `per` = 8, 4, 2 or 1 where many slices give slots
// enough.
__device__ __forceinline__ int64_t sample_row(int64_t i, int shift) {
  // hashed place in the window: cells stored in a repeating order must not alias with it
  const uint32_t x = (uint32_t)i * 2654435761u;
  return (i << shift) + (int64_t)((x >> 16) & ((1u << shift) - 1u));
}

// Resident workgroups per CU of k_bound and k_collect.
template <class Op, int K>
constexpr int scan_minb() {
  if constexpr (Op::kScaled) return K >= 128 ? 3 : 4;
  return K * Op::ESZ <= 128 ? 4 : K * Op::ESZ <= 256 ? 3 : 2;
}

template <class Op, int K>
__global__ void __launch_bounds__(256, (scan_minb<Op, K>())) k_bound(
    const typename Op::Frag *__restrict__ Qp_, int64_t nq, const unsigned char *__restrict__ Rp,
    int64_t m, int shift, int64_t slice_len, int S, int per, float *__restrict__ slot_min) {
  typedef typename Op::Frag Frag;
  constexpr int QG = ScreenShape<Op, K>::QG;
  constexpr int QPW = 32 * QG;
  constexpr int QPB = ScreenShape<Op, K>::QPB;
  constexpr int HALF = K / 2;
  constexpr int NS = HALF / Op::EPL;
  constexpr int GROWB = K * Op::ESZ + (Op::kScaled ? 16 : 0);
  constexpr int ROWB = K * Op::ESZ + 16;
  constexpr int CHUNKS = GROWB / 16;
  constexpr int RT = (2 * 128 * ROWB <= 49152) ? 128 : (2 * 64 * ROWB <= 49152) ? 64 : 32;
  constexpr int CPR = ROWB / 16;
  constexpr int NINSTR = (RT * CPR + 63) / 64;
  constexpr int BUFB = NINSTR * 1024;
  constexpr int JPW = (NINSTR + 3) / 4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_r[2][BUFB];

  const unsigned char *Qp = reinterpret_cast<const unsigned char *>(Qp_);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, n = lane & 31;
  const int slice = blockIdx.y;
  const int64_t r_begin = (int64_t)slice * slice_len;
  const int64_t r_end = min(m, r_begin + slice_len);
  const int qw0 = w * QPW;
  const int64_t qb0 = (int64_t)blockIdx.x * QPB;
  const bool live = qb0 + qw0 < nq;

  Frag bq[QG][NS];
  int qscale[QG];
  float vmin[QG][8];
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const int64_t q = qb0 + qw0 + g * 32 + n;
    qscale[g] = 127;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      bq[g][s] = q < nq ? *reinterpret_cast<const Frag *>(
                              Qp + q * GROWB + (h * HALF + s * Op::EPL) * Op::ESZ)
                        : Frag{};
    if (Op::kScaled && q < nq)
      qscale[g] = *reinterpret_cast<const int32_t *>(Qp + q * GROWB + K * Op::ESZ + 4);
#pragma unroll
    for (int v = 0; v < 8; ++v) vmin[g][v] = INFINITY;
  }

  // stage layout as in k_screen; every chunk's row is looked up, rows past the slice
  // re-read its last one
  auto fetch = [&](int64_t t0, int b) {
#pragma unroll
    for (int i = 0; i < JPW; ++i) {
      const int j = w + 4 * i;
      if (j < NINSTR) {
        const int ci = 64 * j + lane;
        const int rr = ci / CPR, c = ci % CPR;
        const int64_t row = sample_row(min(t0 + rr, r_end - 1), shift);
        __builtin_amdgcn_global_load_lds(
            (const void *)(Rp + row * GROWB + (c < CHUNKS ? c : 0) * 16),
            (__attribute__((address_space(3))) void *)(&lds_r[b][1024 * j]), 16, 0, 0);
      }
    }
  };

  int b = 0;
  if (r_begin < r_end) fetch(r_begin, 0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int64_t t0 = r_begin; t0 < r_end; t0 += RT) {
    if (t0 + RT < r_end) fetch(t0 + RT, b ^ 1);
#pragma unroll 1
    for (int sub = 0; sub < RT / 32; ++sub) {
      const int64_t rb = t0 + sub * 32;
      if (rb >= r_end || !live) break;
      floatx16 acc[QG];
      if constexpr (Op::kScaled) {
        floatx16 nrm;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          nrm[v] = *reinterpret_cast<const float *>(
              &lds_r[b][(sub * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * ROWB + K * Op::ESZ]);
#pragma unroll
        for (int g = 0; g < QG; ++g) acc[g] = nrm;
      } else {
#pragma unroll
        for (int g = 0; g < QG; ++g)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[g][v] = 0.f;
      }
      const unsigned char *arow = &lds_r[b][(sub * 32 + n) * ROWB + h * HALF * Op::ESZ];
      int ascale = 127;
      if constexpr (Op::kScaled)
        ascale = *reinterpret_cast<const int32_t *>(
            &lds_r[b][(sub * 32 + n) * ROWB + K * Op::ESZ + 4]);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        Frag a = *reinterpret_cast<const Frag *>(arow + s * Op::EPL * Op::ESZ);
#pragma unroll
        for (int g = 0; g < QG; ++g) {
          if constexpr (Op::kScaled)
            acc[g] = Op::mma_s(a, bq[g][s], acc[g], ascale, qscale[g]);
          else
            acc[g] = Op::mma(a, bq[g][s], acc[g]);
        }
      }
      if (rb + 32 > r_end) {
#pragma unroll
        for (int g = 0; g < QG; ++g)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (rb + 8 * (v >> 2) + 4 * h + (v & 3) >= r_end) acc[g][v] = INFINITY;
      }
#pragma unroll
      for (int g = 0; g < QG; ++g)
#pragma unroll
        for (int v = 0; v < 8; ++v)
          vmin[g][v] = fminf(fminf(acc[g][2 * v], acc[g][2 * v + 1]), vmin[g][v]);
    }
    __builtin_amdgcn_s_waitcnt(0);  // the next stage's DMA has landed
    __syncthreads();
    b ^= 1;
  }
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const int64_t q = qb0 + qw0 + g * 32 + n;
    if (q >= nq) continue;
    float *o = slot_min + (q * S + slice) * (2 * per) + h * per;
    if (per == 8) {
#pragma unroll
      for (int v = 0; v < 8; ++v) o[v] = vmin[g][v];
    } else if (per == 4) {
#pragma unroll
      for (int v = 0; v < 4; ++v) o[v] = fminf(vmin[g][2 * v], vmin[g][2 * v + 1]);
    } else {
      const float lo = fminf(fminf(vmin[g][0], vmin[g][1]), fminf(vmin[g][2], vmin[g][3]));
      const float hi = fminf(fminf(vmin[g][4], vmin[g][5]), fminf(vmin[g][6], vmin[g][7]));
      if (per == 2) {
        o[0] = lo;
        o[1] = hi;
      } else {
        o[0] = fminf(lo, hi);
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// The scan of all but the smallest searches (pool_plan): k_screen's tile loop against a threshold
// that does not move.
//
// With a threshold per query from k_bound the scan meets a few hundred keys per query, so
// it needs no compaction, no sort and no seeds: a passing key goes to the lane half's
// segment (cap / 2 words of reference index and key bits) and is counted.  k_pool_merge selects
// the pool; a query whose segment overflowed, or that met fewer than `pool` keys (its
// threshold was a guess from a sample), goes on a list and is screened again from an open
// threshold.  A lane half whose segment overflowed collects nothing more: 100,000 cells of
// which half are one row take 6.1 ms in all, with that and k_screen's rule for equal keys (155
// without both, 84 in one scan by a k_screen that inserts them all).  Without the compaction the loop is a tenth of k_screen's code and keeps its
// registers (122 of 128, no spills, against 43 spilled).  262,144 queries x 1,048,576
// references of 64 BF16 elements: 28.0 ms with no key passing (1.26 PFLOP/s; k_screen 31.1),
// 32.3 ms with 213 keys per query.  The loop without filter, LDS reads and staging takes
// 20.2 ms: the matrix cores at the clock that this load leaves them.  Four query groups per
// wave at two workgroups per CU: 25.7 and 32.6 ms, so the smaller block was kept.
template <class Op, int K>
__global__ void __launch_bounds__(256, (scan_minb<Op, K>())) k_collect(
    const typename Op::Frag *__restrict__ Qp_, int64_t nq, const unsigned char *__restrict__ Rp,
    int64_t nr, int64_t slice_len, int S, const float *__restrict__ tau0, int cap,
    uint2 *__restrict__ buf, int32_t *__restrict__ seg_cnt) {
  typedef typename Op::Frag Frag;
  constexpr int QG = ScreenShape<Op, K>::QG;
  constexpr int QPW = 32 * QG;
  constexpr int QPB = ScreenShape<Op, K>::QPB;
  constexpr int HALF = K / 2;
  constexpr int NS = HALF / Op::EPL;
  constexpr int GROWB = K * Op::ESZ + (Op::kScaled ? 16 : 0);
  constexpr int ROWB = K * Op::ESZ + 16;
  constexpr int CHUNKS = GROWB / 16;
  constexpr int RT = (2 * 128 * ROWB <= 49152) ? 128 : (2 * 64 * ROWB <= 49152) ? 64 : 32;
  constexpr int CPR = ROWB / 16;
  constexpr int NINSTR = (RT * CPR + 63) / 64;
  constexpr int BUFB = NINSTR * 1024;
  constexpr int JPW = (NINSTR + 3) / 4;
  constexpr int RROWS = (64 * NINSTR + CPR - 1) / CPR;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_r[2][BUFB];

  const unsigned char *Qp = reinterpret_cast<const unsigned char *>(Qp_);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, n = lane & 31;
  const int slice = blockIdx.y;
  const int64_t r_begin = (int64_t)slice * slice_len;
  const int64_t r_end = min(nr, r_begin + slice_len);
  const int64_t qw = (int64_t)blockIdx.x * QPB + w * QPW;  // wave's first query
  const bool live = qw < nq;
  const int room = cap / 2;

  Frag bq[QG][NS];
  float tau[QG];
  int qscale[QG];
  // write positions: bytes from the wave's first segment; `last` is the segment's last slot,
  // which keys past the room overwrite (the count then says so)
  unsigned char *wbuf = reinterpret_cast<unsigned char *>(buf + (qw * S + slice) * cap);
  uint32_t start[QG], pos[QG], last[QG];
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const int64_t q = qw + g * 32 + n;
    tau[g] = q < nq ? tau0[q] : -INFINITY;  // a query past the batch end never passes
    start[g] = (uint32_t)(((g * 32 + n) * S * cap + h * room) * 8);
    pos[g] = start[g];
    last[g] = start[g] + (uint32_t)(room - 1) * 8;
    qscale[g] = 127;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      bq[g][s] = q < nq ? *reinterpret_cast<const Frag *>(
                              Qp + q * GROWB + (h * HALF + s * Op::EPL) * Op::ESZ)
                        : Frag{};
    if (Op::kScaled && q < nq)
      qscale[g] = *reinterpret_cast<const int32_t *>(Qp + q * GROWB + K * Op::ESZ + 4);
  }

  // stage layout and LDS DMA as in k_screen
  uint32_t choff[JPW];
  int chrow[JPW];
#pragma unroll
  for (int i = 0; i < JPW; ++i) {
    const int ci = 64 * (w + 4 * i) + lane;
    const int rr = ci / CPR, c = ci % CPR;
    chrow[i] = rr;
    choff[i] = (uint32_t)(rr * GROWB + (c < CHUNKS ? c : 0) * 16);
  }
  auto fetch = [&](int64_t t0, int b) {
    const unsigned char *stage = Rp + t0 * GROWB;
    const bool whole = t0 + RROWS <= r_end;
#pragma unroll
    for (int i = 0; i < JPW; ++i) {
      const int j = w + 4 * i;
      if (j < NINSTR) {
        const unsigned char *src = stage + choff[i];
        if (!whole) {  // rows past the slice re-read its last row
          const int64_t last = r_end - 1 - t0;
          src -= (chrow[i] > last ? chrow[i] - last : 0) * GROWB;
        }
        __builtin_amdgcn_global_load_lds(
            (const void *)src,
            (__attribute__((address_space(3))) void *)(&lds_r[b][1024 * j]), 16, 0, 0);
      }
    }
  };

  int b = 0;
  if (r_begin < r_end) fetch(r_begin, 0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int64_t t0 = r_begin; t0 < r_end; t0 += RT) {
    if (t0 + RT < r_end) fetch(t0 + RT, b ^ 1);
    // not unrolled: four copies of the insertion code outgrow the instruction cache's share
#pragma unroll 1
    for (int sub = 0; sub < RT / 32; ++sub) {
      const int64_t rb = t0 + sub * 32;
      if (rb >= r_end || !live) break;
      floatx16 acc[QG];
      if constexpr (Op::kScaled) {
        floatx16 nrm;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          nrm[v] = *reinterpret_cast<const float *>(
              &lds_r[b][(sub * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * ROWB + K * Op::ESZ]);
#pragma unroll
        for (int g = 0; g < QG; ++g) acc[g] = nrm;
      } else {
#pragma unroll
        for (int g = 0; g < QG; ++g)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[g][v] = 0.f;
      }
      const unsigned char *arow = &lds_r[b][(sub * 32 + n) * ROWB + h * HALF * Op::ESZ];
      int ascale = 127;
      if constexpr (Op::kScaled)
        ascale = *reinterpret_cast<const int32_t *>(
            &lds_r[b][(sub * 32 + n) * ROWB + K * Op::ESZ + 4]);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        Frag a = *reinterpret_cast<const Frag *>(arow + s * Op::EPL * Op::ESZ);
#pragma unroll
        for (int g = 0; g < QG; ++g) {
          if constexpr (Op::kScaled)
            acc[g] = Op::mma_s(a, bq[g][s], acc[g], ascale, qscale[g]);
          else
            acc[g] = Op::mma(a, bq[g][s], acc[g]);
        }
      }
      if (rb + 32 > r_end) {  // references past the slice end never pass
#pragma unroll
        for (int g = 0; g < QG; ++g)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (rb + 8 * (v >> 2) + 4 * h + (v & 3) >= r_end) acc[g][v] = INFINITY;
      }
      float m4[QG][4];
      uint64_t hit[QG], any_hit = 0;  // lanes with a passing key, per query group
#pragma unroll
      for (int g = 0; g < QG; ++g) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          m4[g][j] = fminf(fminf(acc[g][4 * j], acc[g][4 * j + 1]),
                           fminf(acc[g][4 * j + 2], acc[g][4 * j + 3]));
        hit[g] = __builtin_amdgcn_ballot_w64(
            fminf(fminf(m4[g][0], m4[g][1]), fminf(m4[g][2], m4[g][3])) <= tau[g]);
        any_hit |= hit[g];
      }
      if (any_hit) {
        const uint32_t ref0 = (uint32_t)(rb + 4 * h);
#pragma unroll
        for (int g = 0; g < QG; ++g) {
          if (!hit[g]) continue;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (wave_any(m4[g][j] <= tau[g])) {
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const float key = acc[g][4 * j + u];
                if (key <= tau[g]) {
                  *reinterpret_cast<uint2 *>(wbuf + min(pos[g], last[g])) =
                      make_uint2(ref0 + (uint32_t)(8 * j + u), __float_as_uint(key));
                  pos[g] += 8;
                }
              }
            }
          }
          // past the room the query is screened again, whatever else it meets
          if ((int)(pos[g] - last[g]) > 8) tau[g] = -INFINITY;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // the next stage's DMA has landed
    __syncthreads();
    b ^= 1;
  }
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const int64_t q = qw + g * 32 + n;
    if (q < nq) seg_cnt[(q * S + slice) * 2 + h] = (int32_t)((pos[g] - start[g]) / 8);
  }
}

// ---------------------------------------------------------------------------------
// Launch interface of one operand type (K: packed row elements, cap: buffer keys).
struct ScreenArgs {
  const void *q;
  int64_t nq;
  const void *r;
  int64_t nr, slice_len;
  int S, pool;
  const int64_t *seeds;   // NULL, or one seed reference per query
  const float *tau0;      // NULL (open), or each query's starting threshold
  const int32_t *list;    // NULL, or the packed rows of the queries: list[list_base + p]
  const int32_t *list_n;  // entries of the list, on the device
  int32_t list_base;
  uint64_t *buf;          // [nq][S][cap]
  int32_t *seg_cnt;       // NULL, or [nq][S][2]: leave the keys in buf, write their counts
  uint64_t *out;          // [nq][S][pool] sorted pools (seg_cnt NULL)
  int32_t *out_cnt;       // [nq][S]
};
struct BoundArgs {
  const void *q;
  int64_t nq;
  const void *r;
  int64_t m;              // sampled rows
  int shift;              // one of each 2^shift rows
  int64_t slice_len;      // sampled rows per slice, a multiple of kSliceAlign
  int S, per;
  float *slot_min;        // [nq][S][2 * per]
};
struct CollectArgs {
  const void *q;
  int64_t nq;
  const void *r;
  int64_t nr, slice_len;
  int S;
  const float *tau0;
  int cap;
  uint2 *buf;        // [nq][S][cap] (index, key bits); 64 * S * cap * 8 bytes fit 32 bits
  int32_t *seg_cnt;  // [nq][S][2], counts past cap / 2 say that keys were dropped
};
struct KnnOps {  // false / 0: no such instantiation
  bool (*screen)(int K, int cap, const ScreenArgs &, hipStream_t);
  bool (*bound)(int K, const BoundArgs &, hipStream_t);
  bool (*collect)(int K, const CollectArgs &, hipStream_t);
  int (*screen_resident)(int K, int cap);  // workgroups per CU
  int (*scan_resident)(int K);
};
KnnOps knn_ops_bf16();
KnnOps knn_ops_fp8();
KnnOps knn_ops_f32();

template <class Op, int K, int CAP>
inline void launch_screen(const ScreenArgs &a, hipStream_t st) {
  dim3 grid((uint32_t)cdiv(a.nq, ScreenShape<Op, K>::QPB), a.S);
  hipLaunchKernelGGL((k_screen<Op, K, CAP>), grid, dim3(256), 0, st,
                     (const typename Op::Frag *)a.q, a.nq, (const unsigned char *)a.r, a.nr,
                     a.slice_len, a.S, a.pool, a.seeds, a.tau0, a.list, a.list_n, a.list_base,
                     a.buf, a.seg_cnt, a.out, a.out_cnt);
}
template <class Op, int K>
inline void launch_collect(const CollectArgs &a, hipStream_t st) {
  dim3 grid((uint32_t)cdiv(a.nq, ScreenShape<Op, K>::QPB), a.S);
  hipLaunchKernelGGL((k_collect<Op, K>), grid, dim3(256), 0, st, (const typename Op::Frag *)a.q,
                     a.nq, (const unsigned char *)a.r, a.nr, a.slice_len, a.S, a.tau0, a.cap,
                     a.buf, a.seg_cnt);
}
template <class Op, int K>
inline void launch_bound(const BoundArgs &a, hipStream_t st) {
  dim3 grid((uint32_t)cdiv(a.nq, ScreenShape<Op, K>::QPB), a.S);
  hipLaunchKernelGGL((k_bound<Op, K>), grid, dim3(256), 0, st, (const typename Op::Frag *)a.q,
                     a.nq, (const unsigned char *)a.r, a.m, a.shift, a.slice_len, a.S, a.per,
                     a.slot_min);
}

// KS: the packed widths this operand type is built for; HUGE: 1,024-key buffers too.
template <class Op, bool HUGE, int... KS>
struct KnnTable {
  template <int K>
  static bool screen_k(int cap, const ScreenArgs &a, hipStream_t st) {
    if (cap == 256)
      launch_screen<Op, K, 256>(a, st);
    else if (cap == 512)
      launch_screen<Op, K, 512>(a, st);
    else if constexpr (HUGE)
      launch_screen<Op, K, 1024>(a, st);
    else
      return false;
    return true;
  }
  static bool screen(int K, int cap, const ScreenArgs &a, hipStream_t st) {
    bool ok = false;
    ((K == KS ? (void)(ok = screen_k<KS>(cap, a, st)) : (void)0), ...);
    return ok;
  }
  static bool bound(int K, const BoundArgs &a, hipStream_t st) {
    bool ok = false;
    ((K == KS ? (launch_bound<Op, KS>(a, st), (void)(ok = true)) : (void)0), ...);
    return ok;
  }
  static bool collect(int K, const CollectArgs &a, hipStream_t st) {
    bool ok = false;
    ((K == KS ? (launch_collect<Op, KS>(a, st), (void)(ok = true)) : (void)0), ...);
    return ok;
  }
  static int screen_resident(int K, int cap) {
    int n = 0;
    ((K == KS ? (void)(n = cap == 256 ? screen_minb<Op, KS, 256>()
                           : cap == 512 ? screen_minb<Op, KS, 512>()
                                        : screen_minb<Op, KS, 1024>())
              : (void)0),
     ...);
    return n;
  }
  static int scan_resident(int K) {
    int n = 0;
    ((K == KS ? (void)(n = scan_minb<Op, KS>()) : (void)0), ...);
    return n;
  }
};

}  // namespace sh
