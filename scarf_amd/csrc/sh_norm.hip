// Library-size normalisation, per-feature statistics, dense z tiles and the sparse
// z-score projection (HBM-bound CSR passes).
//
// Reference semantics (scarf tree): assay.py:41-64 (norm_lib_size[_log]),
// assay.py:812-828 (renormalize_subset library size, 0 -> 1),
// graph_datastore.py:767-796 + utils.py:143-154 (mean/std + clean_array),
// ann.py:129-138 and 191-192 (z-score and reducer).
#include <float.h>

#include <algorithm>
#include <utility>

#include "sh_common.h"
#include "sh_log1p.h"

namespace sh {

// Library size over the mapped columns (exact integers); 0 -> 1.  Sixteen lanes per row, so
// a wave has four rows and up to eight loads a lane in flight; a whole wave per row spent
// its time on three dependent loads and a six-step reduction for some 160 entries.
constexpr int kLibLanes = 16;
__global__ void __launch_bounds__(256) k_libsize(const uint32_t *__restrict__ vals,
                                                 const int32_t *__restrict__ cols,
                                                 const int64_t *__restrict__ rowptr,
                                                 int64_t n_rows,
                                                 const int32_t *__restrict__ col_map,
                                                 int32_t n_in, double *__restrict__ out) {
  const int sub = threadIdx.x % kLibLanes;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / kLibLanes;
  if (row >= n_rows) return;
  const int64_t b = rowptr[row + 1];
  uint64_t s = 0;
#pragma unroll 4
  for (int64_t t = rowptr[row] + sub; t < b; t += kLibLanes) {
    const uint32_t v = vals[t];
    s += map_col(col_map, cols[t], n_in) >= 0 ? v : 0u;
  }
#pragma unroll
  for (int m = kLibLanes / 2; m >= 1; m >>= 1) s += shfl_xor_u64(s, m);
  if (sub == 0) out[row] = s == 0 ? 1.0 : (double)s;
}

// norm_value with the row's 1 / l at hand: the quotient is corrected by its remainder, so it
// is as good as the division (whose 11 instructions, with the library's log1p, were most of
// the statistics), and the logarithm comes from a table in LDS.  What the correction or the
// table is not made for (l = 0, an infinity, next to the ends of the exponent's range) goes
// the general way; inv_l is NaN where 1 / l itself is of no use.
__device__ __forceinline__ double stats_inverse(double l) {
  return l >= 1e-280 && l <= 1e280 ? 1.0 / l : __longlong_as_double(0x7ff8000000000000ll);
}
__device__ __forceinline__ double stats_value(uint32_t v, double sf, double2 l, int log_t,
                                              const LogStep *tab) {
  if (!log_t) return norm_value(v, sf, l.x, 0);
  const double a = sf * (double)v;
  double q = a * l.y;
  q = fma(fma(-q, l.x, a), l.y, q);
  if (q <= 1e300 && (q >= 1e-280 || v == 0)) return log1p_table(q, tab);
  return norm_value(v, sf, l.x, 1);
}

// Per-feature FP64 sums of x and x^2 over a slab of rows, for columns [c0, c0+cb).
// Slabs never straddle a chunk: slab s covers rows [c*chunk + j*slab_rows, ...) of
// chunk c = s / spc, j = s % spc, so every chunk of the matrix is done in one launch.
//
// One workgroup of eight waves per slab.  The slab's non-zeros are a contiguous range of
// the CSR arrays and are streamed flat, one entry per thread and batch with the next
// batch's loads in flight; a thread finds its entry's row by walking the slab's row offsets
// (entries only move forward).  The work is the FP64 division and log1p of every entry, and
// what bounded a form with one wave per accumulator was latency: the accumulators (32 KB at
// 2000 features) left one wave per SIMD.  Here eight waves share them: all normalise, into
// a double-buffered batch in LDS, and one wave at a time, in turn, adds a finished batch
// while the others are at the next.  Batches are added in order, one wave's ds_add lanes
// meet in a fixed order, so the sums are bitwise reproducible.
// 500,000 x 2000 at 8% non-zeros: 1455 -> 551 us; 5,000 rows: 626 -> 20 us.  Counters then
// showed 189 vector instructions for 64 entries, three quarters of the time: the corrected quotient
// and the table (stats_value) took it to 400 us.  The two LDS f64 adds are 105 us of LDS time
// (23 clocks a wave instruction at random features, 8 at consecutive ones).  The batches wait
// for the wave that adds, so it reads its eight pieces before the first add: 356 us (two waves,
// one for the squares: 380, they read twice); a thread keeps its row's end in a register: 347.
// Library sizes summed in here instead of by k_libsize: 601 against 400 + 195, since all
// workgroups are in that phase at the same time.
constexpr int kStatsThreads = 512;
constexpr int kStatsResident = 3 * 256;   // workgroups that fit the GPU (LDS)
constexpr int kStatsMinRows = 16, kStatsMaxRows = 384;  // rows per slab
__global__ void __launch_bounds__(kStatsThreads, 6) k_norm_stats(
    const uint32_t *__restrict__ vals, const int32_t *__restrict__ cols,
    const int64_t *__restrict__ rowptr, int64_t n_rows, int64_t chunk_rows, int spc,
    int64_t slab_rows, const int32_t *__restrict__ col_map, int32_t n_in, int32_t d,
    int32_t cb, double sf, int log_t, const double *__restrict__ libsize,
    double *__restrict__ part /* [n_slabs][2][d] */) {
  // [2][cb], (library size, 1 / it) [slab_rows]
  extern __shared__ __attribute__((aligned(16))) double acc[];
  __shared__ LogStep slog[kLogSteps];
  __shared__ double bx[2][kStatsThreads];
  __shared__ int16_t bf[2][kStatsThreads];  // column within the block, -1: none
  __shared__ int32_t srp[kStatsMaxRows + 1];
  double2 *sls = reinterpret_cast<double2 *>(acc + 2 * cb);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int32_t c0 = blockIdx.y * cb;
  const int32_t ncol = min(d, c0 + cb) - c0;
  const int64_t chunk = blockIdx.x / spc, j_in = blockIdx.x % spc;
  const int64_t c_end = min(n_rows, (chunk + 1) * chunk_rows);
  const int64_t r0 = chunk * chunk_rows + j_in * slab_rows;
  // the last chunk can be shorter than spc slabs: its trailing slabs are empty
  const int nrow = (int)max<int64_t>(0, min(c_end, r0 + slab_rows) - r0);
  const int64_t e0 = nrow > 0 ? rowptr[r0] : 0;
  for (int i = tid; i < 2 * cb; i += kStatsThreads) acc[i] = 0.0;
  for (int i = tid; i <= nrow; i += kStatsThreads)
    srp[i] = nrow > 0 ? (int32_t)(rowptr[r0 + i] - e0) : 0;
  for (int i = tid; i < nrow; i += kStatsThreads) {
    const double l = libsize[r0 + i];
    sls[i] = make_double2(l, stats_inverse(l));
  }
  if (tid < kLogSteps) slog[tid] = kLogTable[tid];
  __syncthreads();
  const int32_t total = srp[nrow];
  const uint32_t *sv = vals + e0;
  const int32_t *sc = cols + e0;
  auto add = [&](int b) {
    int f[kStatsThreads / 64];
    double x[kStatsThreads / 64];
#pragma unroll
    for (int g = 0; g < kStatsThreads / 64; ++g) {
      f[g] = bf[b][64 * g + lane];
      x[g] = bx[b][64 * g + lane];
    }
#pragma unroll
    for (int g = 0; g < kStatsThreads / 64; ++g) {
      if (f[g] >= 0) {
        atomicAdd(&acc[f[g]], x[g]);
        atomicAdd(&acc[cb + f[g]], x[g] * x[g]);
      }
    }
  };
  int row = 0;  // slab-relative row of this thread's current entry
  int32_t row_end = nrow > 0 ? srp[1] : 0;
  uint32_t v = 0;
  int32_t c = -1;
  if (tid < total) {
    v = sv[tid];
    c = sc[tid];
  }
  int batch = 0;
  for (int32_t base = 0; base < total; base += kStatsThreads, ++batch) {
    const int32_t e = base + tid;
    uint32_t vn = 0;
    int32_t cn = -1;
    if (e + kStatsThreads < total) {
      vn = sv[e + kStatsThreads];
      cn = sc[e + kStatsThreads];
    }
    if (batch > 0 && w == ((batch - 1) & 7)) add((batch - 1) & 1);
    int f = -1;
    double x = 0.0;
    if (e < total) {
      while (row_end <= e) row_end = srp[++row + 1];
      f = map_col(col_map, c, n_in) - c0;
      if (f >= 0 && f < ncol)
        x = stats_value(v, sf, sls[row], log_t, slog);
      else
        f = -1;
    }
    bf[batch & 1][tid] = (int16_t)f;
    bx[batch & 1][tid] = x;
    __syncthreads();
    v = vn;
    c = cn;
  }
  if (batch > 0 && w == ((batch - 1) & 7)) add((batch - 1) & 1);
  __syncthreads();
  double *dst = part + (size_t)blockIdx.x * 2 * d;
  for (int j = tid; j < ncol; j += kStatsThreads) {
    dst[c0 + j] = acc[j];
    dst[d + c0 + j] = acc[cb + j];
  }
}

// The chunk's slabs summed in a fixed order: eight interleaved sums per (chunk, feature), one
// thread each, and then those (short rounding chains, and eight times the loads in flight:
// with one thread for all of a chunk's 230 slabs this took 194 us of a 930 us pass).
constexpr int kRedFeat = 32, kRedPart = 8;
__global__ void __launch_bounds__(kRedFeat *kRedPart) k_reduce_slabs(
    const double *__restrict__ part, int spc, int32_t d, double *__restrict__ sum_out,
    double *__restrict__ sq_out) {
  __shared__ double ss[kRedPart][kRedFeat], sq[kRedPart][kRedFeat];
  const int tf = threadIdx.x % kRedFeat, u = threadIdx.x / kRedFeat;
  const int32_t f = (int32_t)blockIdx.x * kRedFeat + tf;
  const int64_t c = blockIdx.y;
  double s = 0.0, q = 0.0;
  if (f < d) {
#pragma unroll 4
    for (int i = u; i < spc; i += kRedPart) {
      const size_t base = (size_t)(c * spc + i) * 2 * d;
      s += part[base + f];
      q += part[base + d + f];
    }
  }
  ss[u][tf] = s;
  sq[u][tf] = q;
  __syncthreads();
  if (u == 0 && f < d) {
    sum_out[c * d + f] = ((ss[0][tf] + ss[1][tf]) + (ss[2][tf] + ss[3][tf])) +
                         ((ss[4][tf] + ss[5][tf]) + (ss[6][tf] + ss[7][tf]));
    sq_out[c * d + f] = ((sq[0][tf] + sq[1][tf]) + (sq[2][tf] + sq[3][tf])) +
                        ((sq[4][tf] + sq[5][tf]) + (sq[6][tf] + sq[7][tf]));
  }
}

// clean_array (utils.py:143-154): nan_to_num maps NaN -> 0 and +-inf -> +-DBL_MAX
// first, so the later "+-inf -> 0" step never fires; then 0 -> fill.
__device__ __forceinline__ double clean(double v, double fill) {
  if (!(v == v)) v = 0.0;
  else if (isinf(v)) v = v > 0 ? DBL_MAX : -DBL_MAX;
  return v == 0.0 ? fill : v;
}

// Chan et al. pairwise merge of per-chunk (n, mean, M2), chunk order fixed.
__global__ void k_stats_merge(const double *__restrict__ sums, const double *__restrict__ sqs,
                              const int64_t *__restrict__ counts, int32_t n_chunks, int32_t d,
                              double *__restrict__ mu, double *__restrict__ sigma,
                              double *__restrict__ chunk_mean) {
  int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= d) return;
  double n = 0.0, mean = 0.0, m2 = 0.0;
  for (int c = 0; c < n_chunks; ++c) {
    double nc = (double)counts[c];
    if (nc <= 0) {
      if (chunk_mean) chunk_mean[(size_t)c * d + f] = 0.0;
      continue;
    }
    double s = sums[(size_t)c * d + f], q = sqs[(size_t)c * d + f];
    double mc = s / nc;
    double m2c = q - s * mc;
    if (m2c < 0) m2c = 0;
    if (chunk_mean) chunk_mean[(size_t)c * d + f] = mc;
    double nn = n + nc;
    double delta = mc - mean;
    mean += delta * (nc / nn);
    m2 += m2c + delta * delta * (n * nc / nn);
    n = nn;
  }
  double var = n > 0 ? m2 / n : 0.0;
  mu[f] = clean(n > 0 ? mean : 0.0, 0.0);
  sigma[f] = clean(sqrt(var), 1.0);
}

// One workgroup per row batch: the dense row is assembled in LDS, then streamed out.
template <typename T>
__global__ void __launch_bounds__(256) k_densify(
    const uint32_t *__restrict__ vals, const int32_t *__restrict__ cols,
    const int64_t *__restrict__ rowptr, const int64_t *__restrict__ rows, int64_t n_rows,
    const int32_t *__restrict__ col_map, int32_t n_in, int32_t d, double sf, int log_t,
    const double *__restrict__ libsize, const double *__restrict__ center,
    const double *__restrict__ scale, double clip, T *__restrict__ out, int64_t ld,
    int rows_per_block) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dbuf_raw[];
  T *buf = reinterpret_cast<T *>(dbuf_raw);  // [ld]
  const int64_t rb = (int64_t)blockIdx.x * rows_per_block;
  for (int rr = 0; rr < rows_per_block; ++rr) {
    const int64_t i = rb + rr;
    if (i >= n_rows) break;
    const int64_t r = rows ? rows[i] : i;
    for (int64_t f = threadIdx.x; f < ld; f += blockDim.x) {
      double v = f == d ? 1.0 : 0.0;  // column d (padding) holds ones: Z^T Z gets column sums
      if (f < d) {
        v = (0.0 - center[f]) * scale[f];
        if (clip > 0.0) v = fmin(fmax(v, -clip), clip);
      }
      buf[f] = (T)v;
    }
    __syncthreads();
    const int64_t a = rowptr[r], b = rowptr[r + 1];
    const double l = libsize[r];
    for (int64_t t = a + threadIdx.x; t < b; t += blockDim.x) {
      int f = map_col(col_map, cols[t], n_in);
      if (f >= 0) {
        double x = norm_value(vals[t], sf, l, log_t);
        double v = (x - center[f]) * scale[f];
        if (clip > 0.0) v = fmin(fmax(v, -clip), clip);
        buf[f] = (T)v;
      }
    }
    __syncthreads();
    float4 *o4 = reinterpret_cast<float4 *>(out + i * ld);
    const float4 *b4 = reinterpret_cast<const float4 *>(buf);
    const int64_t n16 = ld * (int64_t)sizeof(T) / 16;
    for (int64_t f = threadIdx.x; f < n16; f += blockDim.x) o4[f] = b4[f];
    __syncthreads();
  }
}

// Sparse projection E[r] = c + sum over the row's non-zeros of (z(x) - z(0)) W[f]
// (c, the projection of an all-zero row, is precomputed by the caller).  One wave per
// row.  A batch of 64 non-zeros is normalised lane-parallel (x in FP32 from log1pf, the
// z-delta, the mapped feature); the wave's four 16-lane groups then take every fourth
// entry, and lane c of a group loads columns 4c..4c+3 of that entry's W row with one
// 16-byte load (W rows padded to a multiple of 4 floats) and adds delta * W into four
// FP32 accumulators.  Each group thus gathers a whole W row per load instruction; the
// groups' sums are added in a fixed order at the end of the row.  DPL = 64-column
// passes (D <= 64 * DPL).
//
// A group's own lanes hold its entries (lane i of group g: entry 4 i + g of the batch), so an
// entry reaches its group by a DPP row broadcast, which for W's address is part of the add;
// the normalised value of a count below 64 comes from lane `count` of a per-row table, since
// most counts are small and log1pf is 70 instructions; the next batch's counts are in flight
// during this one's gathers.  Together that took the vector instructions from 477 to 324
// million at 500,000 x 2000 with 8% non-zeros and D = 50, and the time from 1327 to 1298 us:
// what bounds it there is the L1's share of the gathers (16.6 GB).  k_project_hot takes them
// from LDS.
constexpr int kProjGroup = 16;
template <int I>
__device__ __forceinline__ int row_bcast(int v) {  // lane I of each 16-lane row
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + I, 0xF, 0xF, true);
}
// library size over the mapped columns (the mapping target's), for the whole wave
__device__ __forceinline__ double mapped_libsize(const uint32_t *vals, const int32_t *cols,
                                                 int64_t a, int64_t b, const int32_t *col_map,
                                                 int32_t n_in, int lane) {
  uint64_t s = 0;
  for (int64_t t = a + lane; t < b; t += 64)
    if (map_col(col_map, cols[t], n_in) >= 0) s += vals[t];
  s = wave_sum_u64(s);
  return s == 0 ? 1.0 : (double)s;
}
// normalised value of a count below 64, lane v's for count v
__device__ __forceinline__ float project_lut(float scale, int log_t, int lane) {
  const float x = (float)lane * scale;
  return log_t ? log1pf(x) : x;
}
// an entry's feature (-1: none) and what its W row is multiplied by
__device__ __forceinline__ float project_delta(uint32_t v, int32_t c, bool there, float lut,
                                               float scale, int log_t, const int32_t *col_map,
                                               int32_t n_in, const float *mu,
                                               const float *inv_sigma, int stride, float clip,
                                               int *feature) {
  float xv = __int_as_float(
      __builtin_amdgcn_ds_bpermute((int)(min(v, 63u) << 2), __float_as_int(lut)));
  const int f = there ? map_col(col_map, c, n_in) : -1;
  *feature = f;
  if (f < 0) return 0.f;
  if (v > 63u) {
    const float x = (float)v * scale;
    xv = log_t ? log1pf(x) : x;
  }
  const float is = inv_sigma[f * stride];
  if (clip > 0.f) {
    const float m = mu[f * stride];
    const float zs = (xv - m) * is;
    const float z0 = (0.f - m) * is;
    return fminf(fmaxf(zs, -clip), clip) - fminf(fmaxf(z0, -clip), clip);
  }
  return xv * is;
}
// steps (of four entries) whose loads are all in flight before the first is used; with two loads a
// step half of that, since the registers of eight leave a SIMD four waves instead of six, but
// where a launch is at most two fills of those (us with eight / four steps at D = 128: 1000 x 2000
// at 8% 16.7 / 19, 100,000 at 2% 147 / 126, 300,000 at 0.5% 299 / 231, at 8% 1229 / 1230; with
// library sizes in the kernel 23.7 / 26.9, 167 / 136, 358 / 268, 1409 / 1198)
constexpr int kProjSteps = 8;
constexpr int64_t kProjFewRows = 256 * 32;
// W's address for a lane: `at` is the entry's byte offset (its row index if WIDE), `lo` the
// lane's own
template <bool WIDE>
__device__ __forceinline__ float4 project_load(int at, uint32_t lo, const char *W,
                                               int64_t row_bytes) {
  if (WIDE) return *reinterpret_cast<const float4 *>(W + (int64_t)at * row_bytes + lo);
  return *reinterpret_cast<const float4 *>(W + ((uint32_t)at + lo));
}
template <int DPL>
__device__ __forceinline__ void project_add(float dj, const float4 (&w)[DPL], float4 (&acc)[DPL]) {
#pragma unroll
  for (int p = 0; p < DPL; ++p) {
    acc[p].x = fmaf(dj, w[p].x, acc[p].x);
    acc[p].y = fmaf(dj, w[p].y, acc[p].y);
    acc[p].z = fmaf(dj, w[p].z, acc[p].z);
    acc[p].w = fmaf(dj, w[p].w, acc[p].w);
  }
}
// Entries that are none (behind the row's end, or of a feature that is not taken) are masked,
// in scalar instructions; a block without any skips that.  0 * 0 is added for them: W itself
// may hold an infinity.
template <int DPL, bool WIDE, int B, int... I>
__device__ __forceinline__ void project_steps(std::integer_sequence<int, I...>, int at,
                                              float delta, uint64_t valid,
                                              const uint32_t (&lo)[DPL], const char *W,
                                              int64_t row_bytes, float4 (&acc)[DPL]) {
  constexpr uint64_t kStep = 0x0001000100010001ull;  // lane 0 of each group
  constexpr uint64_t kAll = (((1ull << sizeof...(I)) - 1) << B) * kStep;
  float4 w[sizeof...(I)][DPL];
  if ((valid & kAll) == kAll) {
    (
        [&] {
#pragma unroll
          for (int p = 0; p < DPL; ++p)
            w[I][p] = project_load<WIDE>(row_bcast<B + I>(at), lo[p], W, row_bytes);
        }(),
        ...);
  } else {
    (
        [&] {
          const uint64_t m = (valid >> (B + I)) & kStep;
#pragma unroll
          for (int p = 0; p < DPL; ++p) w[I][p] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (__builtin_amdgcn_inverse_ballot_w64((m << 16) - m)) {
#pragma unroll
            for (int p = 0; p < DPL; ++p)
              w[I][p] = project_load<WIDE>(row_bcast<B + I>(at), lo[p], W, row_bytes);
          }
        }(),
        ...);
  }
  (project_add<DPL>(__int_as_float(row_bcast<B + I>(__float_as_int(delta))), w[I], acc), ...);
}
// groups 0 + 1 and 2 + 3, then the two pairs
template <int DPL>
__device__ __forceinline__ void project_store(float4 (&acc)[DPL], const bool (&col_ok)[DPL],
                                              int grp, int c4, int32_t D, const float *cvec,
                                              float *e) {
  const int lane = grp * kProjGroup + c4;
  auto from = [](int l, float x) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(l << 2, __float_as_int(x)));
  };
  auto add = [&](int l, float4 &x) {
    x = make_float4(x.x + from(l, x.x), x.y + from(l, x.y), x.z + from(l, x.z),
                    x.w + from(l, x.w));
  };
#pragma unroll
  for (int p = 0; p < DPL; ++p) {
    add(lane ^ 16, acc[p]);
    add(lane ^ 32, acc[p]);
    const int col = 4 * (c4 + kProjGroup * p);
    if (grp == 0 && col_ok[p]) {
      float *o = e + col;
      o[0] = acc[p].x + cvec[col];
      if (col + 1 < D) o[1] = acc[p].y + cvec[col + 1];
      if (col + 2 < D) o[2] = acc[p].z + cvec[col + 2];
      if (col + 3 < D) o[3] = acc[p].w + cvec[col + 3];
    }
  }
}
template <int DPL, bool WIDE, int STEPS>
__global__ void __launch_bounds__(256) k_project(
    const uint32_t *__restrict__ vals, const int32_t *__restrict__ cols,
    const int64_t *__restrict__ rowptr, int64_t n_rows, const int32_t *__restrict__ col_map,
    int32_t n_in, float sf, int log_t, const double *__restrict__ libsize,
    const float *__restrict__ mu, const float *__restrict__ inv_sigma, float clip,
    const float *__restrict__ W, int64_t ldw, int32_t D, const float *__restrict__ cvec,
    float *__restrict__ E, int64_t lde) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= n_rows) return;
  const int grp = lane / kProjGroup, c4 = lane % kProjGroup;
  const int64_t a = rowptr[row], b = rowptr[row + 1];
  const float scale =
      sf / (float)(libsize ? libsize[row] : mapped_libsize(vals, cols, a, b, col_map, n_in, lane));
  const char *Wb = reinterpret_cast<const char *>(W);
  const int64_t row_bytes = ldw * 4;
  // lanes past a row's last columns load them again and store nothing
  bool col_ok[DPL];
  uint32_t lo[DPL];
#pragma unroll
  for (int p = 0; p < DPL; ++p) {
    const int c = c4 + kProjGroup * p;
    col_ok[p] = 4 * c < D;
    lo[p] = 16u * (uint32_t)min(c, (D - 1) / 4);
  }
  const float lut = project_lut(scale, log_t, lane);
  float4 acc[DPL];
#pragma unroll
  for (int p = 0; p < DPL; ++p) acc[p] = make_float4(0.f, 0.f, 0.f, 0.f);
  const int mine = 4 * c4 + grp;  // this lane's entry of a batch
  int32_t c = -1;
  uint32_t v = 0;
  if (a + mine < b) {
    c = cols[a + mine];
    v = vals[a + mine];
  }
  for (int64_t t0 = a; t0 < b; t0 += 64) {
    const int64_t tn = t0 + 64 + mine;
    int32_t cn = -1;
    uint32_t vn = 0;
    if (tn < b) {
      cn = cols[tn];
      vn = vals[tn];
    }
    int f;
    const float delta = project_delta(v, c, t0 + mine < b, lut, scale, log_t, col_map, n_in, mu,
                                      inv_sigma, 1, clip, &f);
    const uint64_t valid = __ballot(f >= 0);
    const int at = WIDE ? f : (int)((uint32_t)f * (uint32_t)row_bytes);
    const auto seq = std::make_integer_sequence<int, STEPS>{};
    project_steps<DPL, WIDE, 0>(seq, at, delta, valid, lo, Wb, row_bytes, acc);
    if (b - t0 > 4 * STEPS)
      project_steps<DPL, WIDE, STEPS>(seq, at, delta, valid, lo, Wb, row_bytes, acc);
    if constexpr (STEPS == 4) {
      if (b - t0 > 8 * STEPS)
        project_steps<DPL, WIDE, 2 * STEPS>(seq, at, delta, valid, lo, Wb, row_bytes, acc);
      if (b - t0 > 12 * STEPS)
        project_steps<DPL, WIDE, 3 * STEPS>(seq, at, delta, valid, lo, Wb, row_bytes, acc);
    }
    c = cn;
    v = vn;
  }
  project_store<DPL>(acc, col_ok, grp, c4, D, cvec, E + row * lde);
}

// The same projection with the rows of W that are used most in LDS: one workgroup of 16 waves
// a CU for the whole launch.  Non-zeros are uneven over features (of 2000 features the 700 most
// used hold about 80% of them), and LDS gives a row twice as fast as L1 and without L2 behind
// it.  Which rows those are does not change a result, so each workgroup chooses by itself, from
// the features it counts in kHotSample rows of each wave (2, 8, 16, 32, 64: 984, 990, 1005,
// 1030, 1078 us against 990 with 4).  LDS also holds mean and 1 / sigma (gathered from L1 they
// cost 115 us) and each feature's place in the table.  An entry reads the table's row, or its
// row of zeros, and then, under a mask of the groups that have one, W's row in global memory
// over it; both halves of a batch are in flight at once, and during them the next batch is
// normalised.  A wave reads the bounds and scales of 64 rows at once and a row's first batches
// during the row before, so no row waits for a chain of loads.  The additions and their order
// are those of k_project.
//
// 500,000 x 2000 at 8%, D = 50: 1298 -> 855 us (930 under a profiler).  Without the masked
// loads it would be about 670, and about 460 without any gather: what is left is shared
// between the row's own reads, vector instructions (about 0.45 ms of them) and L2 latency of
// the last 20%.
constexpr int kHotLds = 158 * 1024;    // of a CU's 160 KB
constexpr uint16_t kHotNone = 0xffff;  // a feature whose row is not in the table
constexpr int kHotThreads = 1024;
constexpr int kHotBlocks = 256;  // one a CU
constexpr int kHotSample = 4;    // rows a wave samples for the counts
// Building the table costs 15-70 us a launch, more with more features, so it takes 32 rows a
// wave to pay: at 8% non-zeros and 131,072 rows 111 us against 108 at 600 features and 8%, 145 / 157 at 1000,
// 239 / 279 at 2000, 511 / 700 at 4000 (8%) and 527 / 699 at 6000, 746 / 923 at 8000 (5%); at
// half as many rows 64 / 58, 139 / 148, 261 / 291.  Beyond 8192 features the means and places
// leave less than half of LDS to the table.
constexpr int64_t kHotRows = (int64_t)kHotBlocks * (kHotThreads / 64) * 32;
constexpr int kHotMaxD = 8192;
// A row costs more too (1.1 ns against 0.45 in k_project, where 32 waves a CU share the row's own
// loads instead of 16; 0.7 against 0.35 if the library sizes are given) and an entry less, so rows
// have to be long enough, where the caller says how long they are.  us with the table / without,
// 2000 features, library sizes given: 500,000 rows of 10 entries 292 / 241, of 40 420 / 415, of 80
// 610 / 769; 131,072 rows of 40 117 / 103, of 80 162 / 167, of 160 255 / 295.  Summed in the
// kernel: 500,000 rows of 40 563 / 472, of 80 847 / 910; 131,072 of 80 218 / 195, of 160 342 / 341.
constexpr bool hot_entries(int64_t n_rows, int64_t entries, bool libsize) {
  return entries >= (libsize ? 28 * n_rows + 4000000 : 60 * n_rows + 8000000);
}

// explicitly LDS: through a generic pointer the compiler joins the two sources of an entry's
// row into one flat load
typedef const __attribute__((address_space(3))) char *LdsBytes;
__device__ __forceinline__ float4 lds_float4(LdsBytes p, uint32_t at) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 x = *(const __attribute__((address_space(3))) f4 *)(p + at);
  return make_float4(x.x, x.y, x.z, x.w);
}
// an entry of a batch on its lane: what its row is multiplied by, where that is in the table
// (the row of zeros if nowhere) and in W, in bytes; and the wave's entries not in the table
struct HotEntry {
  float delta;
  int hat, at;
  uint64_t cold;
};
template <int B, int... I>
__device__ __forceinline__ void hot_gather(std::integer_sequence<int, I...>, const HotEntry &e,
                                           uint32_t lo, LdsBytes tab, const char *W,
                                           float4 (&w)[kProjSteps][1]) {
  constexpr uint64_t kStep = 0x0001000100010001ull;  // lane 0 of each group
  ((w[I][0] = lds_float4(tab, (uint32_t)row_bcast<B + I>(e.hat) + lo)), ...);
  (
      [&] {
        const uint64_t m = (e.cold >> (B + I)) & kStep;
        if (__builtin_amdgcn_inverse_ballot_w64((m << 16) - m))
          w[I][0] = project_load<false>(row_bcast<B + I>(e.at), lo, W, 0);
      }(),
      ...);
}
template <int B, int... I>
__device__ __forceinline__ void hot_add(std::integer_sequence<int, I...>, float delta,
                                        const float4 (&w)[kProjSteps][1], float4 (&acc)[1]) {
  (project_add<1>(__int_as_float(row_bcast<B + I>(__float_as_int(delta))), w[I], acc), ...);
}
constexpr int kProjQueue = 4;  // batches of a row loaded ahead
struct ProjQueue {
  int32_t c[kProjQueue];
  uint32_t v[kProjQueue];
  // the first batches of a row of n entries
  __device__ __forceinline__ void load(const uint32_t *vals, const int32_t *cols, int n, int mine) {
#pragma unroll
    for (int i = 0; i < kProjQueue; ++i) fetch(i, vals, cols, 64 * i, n, mine);
  }
  __device__ __forceinline__ void fetch(int i, const uint32_t *vals, const int32_t *cols, int t,
                                        int n, int mine) {
    c[i] = -1;
    v[i] = 0;
    if (t + mine < n) {
      c[i] = cols[t + mine];
      v[i] = vals[t + mine];
    }
  }
  // drop the first batch and load the one that starts at entry t
  __device__ __forceinline__ void next(const uint32_t *vals, const int32_t *cols, int t, int n,
                                       int mine) {
#pragma unroll
    for (int i = 0; i + 1 < kProjQueue; ++i) {
      c[i] = c[i + 1];
      v[i] = v[i + 1];
    }
    if (t < n) fetch(kProjQueue - 1, vals, cols, t, n, mine);
  }
};
__device__ __forceinline__ int64_t lane_i64(int64_t x, int i) {
  return (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, i) |
         ((int64_t)__builtin_amdgcn_readlane((int)(x >> 32), i) << 32);
}
template <bool MAPPED>
__global__ void __launch_bounds__(kHotThreads) k_project_hot(
    const uint32_t *__restrict__ vals, const int32_t *__restrict__ cols,
    const int64_t *__restrict__ rowptr, int64_t n_rows, const int32_t *__restrict__ map,
    int32_t n_in, int32_t d, float sf, int log_t, const double *__restrict__ libsize,
    const float *__restrict__ mu, const float *__restrict__ inv_sigma, float clip,
    const float *__restrict__ W, int64_t ldw, int32_t D, const float *__restrict__ cvec,
    float *__restrict__ E, int64_t lde) {
  __shared__ float4 mem[kHotLds / 16];
  const int32_t *col_map = MAPPED ? map : nullptr;
  constexpr int kWaves = kHotThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = lane / kProjGroup, c4 = lane % kProjGroup;
  const uint32_t ld4 = (uint32_t)(ldw / 4);
  const uint32_t td4 = (uint32_t)(D + 3) / 4;  // the table's rows are packed
  const int slot4 = (d + 7) / 8 + (d + 1) / 2;  // the slots' and (mean, 1 / sigma) pairs' share
  const int hot = (kHotLds / 16 - 32 - slot4) / (int)td4 - 1;  // and a row of zeros
  int *red = reinterpret_cast<int *>(mem);  // 2 x 16 wave counts, a cursor
  uint16_t *slot = reinterpret_cast<uint16_t *>(mem + 32);
  float2 *mi = reinterpret_cast<float2 *>(mem + 32 + (d + 7) / 8);
  float4 *tab = mem + 32 + slot4;
  uint32_t *hist = reinterpret_cast<uint32_t *>(tab);
  const float4 *W4 = reinterpret_cast<const float4 *>(W);
  const int64_t rstep = (int64_t)gridDim.x * kWaves;
  const int64_t row0 = (int64_t)blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(wave);

  // counts over the sample
  for (int f = tid; f < d; f += kHotThreads) {
    hist[f] = 0;
    mi[f] = make_float2(mu[f], inv_sigma[f]);
  }
  if (tid == 0) red[32] = 0;
  __syncthreads();
  const int64_t mine_rows = row0 < n_rows ? (n_rows - row0 + rstep - 1) / rstep : 0;
  for (int q = 0; q < kHotSample; ++q) {
    const int64_t k = mine_rows * q / kHotSample;
    if (mine_rows > 0) {
      const int64_t r = row0 + k * rstep;
      const int64_t a = rowptr[r], b = rowptr[r + 1];
      for (int64_t t = a + lane; t < b; t += 64) {
        const int f = map_col(col_map, cols[t], n_in);
        if (f >= 0 && f < d) atomicAdd(&hist[f], 1u);
      }
    }
  }
  __syncthreads();
  // the smallest count that at most `hot` features reach; those of the count below it fill up
  uint32_t under = 0, least = 1;
  bool fits = d <= hot;
  if (!fits) {
    int par = 0;
    auto reach = [&](uint32_t T) {
      int n = 0;
      for (int f = tid; f < d; f += kHotThreads) n += hist[f] >= T;
      for (int m = 32; m >= 1; m >>= 1) n += __shfl_xor(n, m, 64);
      if (lane == 0) red[par * 16 + wave] = n;
      __syncthreads();
      n = 0;
      for (int i = 0; i < kWaves; ++i) n += red[par * 16 + i];
      par ^= 1;
      return n;
    };
    while (least < 0x40000000u && reach(least) > hot) {
      under = least;
      least *= 2;
    }
    while (least - under > 1) {
      const uint32_t mid = under + (least - under) / 2;
      if (reach(mid) > hot)
        under = mid;
      else
        least = mid;
    }
  }
  __syncthreads();
  for (int pass = 0; pass < 2; ++pass) {
    for (int f = tid; f < d; f += kHotThreads) {
      const uint32_t h = hist[f];
      if (fits) {
        if (pass == 0) slot[f] = (uint16_t)(f * td4);
      } else if (pass == 0 ? h >= least : h == under) {
        const int q = atomicAdd(&red[32], 1);
        slot[f] = q < hot ? (uint16_t)(q * (int)td4) : kHotNone;
      } else if (pass == 0) {
        slot[f] = kHotNone;
      }
    }
    __syncthreads();
  }
  for (int f = wave * 4 + grp; f < d; f += kWaves * 4) {
    const int q = slot[f];
    if (q == kHotNone) continue;
    for (uint32_t c = c4; c < td4; c += kProjGroup) tab[q + c] = W4[(uint64_t)f * ld4 + c];
  }
  if (tid < (int)td4) tab[hot * td4 + tid] = make_float4(0.f, 0.f, 0.f, 0.f);
  __syncthreads();

  const uint32_t zero = (uint32_t)hot * td4;  // the row of zeros
  const char *Wb = reinterpret_cast<const char *>(W);
  const LdsBytes tb = (LdsBytes)(reinterpret_cast<const char *>(tab));
  const bool col_ok[1] = {4 * c4 < D};
  const uint32_t lo = 16u * (uint32_t)min(c4, (D - 1) / 4);
  const int mine = 4 * c4 + grp;
  for (int64_t k0 = 0; k0 < mine_rows; k0 += 64) {
    // lane i: the bounds and the scale of this wave's row k0 + i
    int64_t A = 0, B = 0;
    float S = 0.f;
    if (k0 + lane < mine_rows) {
      const int64_t r = row0 + (k0 + lane) * rstep;
      A = rowptr[r];
      B = rowptr[r + 1];
      if (libsize) S = sf / (float)libsize[r];
    }
    const int n_here = (int)min<int64_t>(64, mine_rows - k0);
    ProjQueue q, nq;
    int64_t a = lane_i64(A, 0);
    int n = (int)(lane_i64(B, 0) - a);
    q.load(vals + a, cols + a, n, mine);
    for (int i = 0; i < n_here; ++i) {
      const int64_t row = row0 + (k0 + i) * rstep;
      const int ni = min(i + 1, n_here - 1);
      const int64_t na = lane_i64(A, ni);
      const int nn = (int)(lane_i64(B, ni) - na);
      nq.load(vals + na, cols + na, nn, mine);
      const float scale =
          libsize ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(S), i))
                  : sf / (float)mapped_libsize(vals, cols, a, a + n, col_map, n_in, lane);
      const float lut = project_lut(scale, log_t, lane);
      float4 acc[1] = {make_float4(0.f, 0.f, 0.f, 0.f)};
      auto entry = [&](int t0) {
        HotEntry e;
        int f;
        e.delta = project_delta(q.v[0], q.c[0], t0 + mine < n, lut, scale, log_t, col_map, n_in,
                                &mi[0].x, &mi[0].y, 2, clip, &f);
        const uint32_t at_slot = f >= 0 ? slot[f] : zero;
        e.cold = __ballot(at_slot == kHotNone);
        e.hat = 16 * (int)(at_slot == kHotNone ? zero : at_slot);
        e.at = (int)((uint32_t)f * 4u * (uint32_t)ldw);
        return e;
      };
      HotEntry e = entry(0);
      for (int t0 = 0; t0 < n; t0 += 64) {
        const auto seq = std::make_integer_sequence<int, kProjSteps>{};
        float4 w[kProjSteps][1], x[kProjSteps][1];
        HotEntry en = e;
        hot_gather<0>(seq, e, lo, tb, Wb, w);
        if (n - t0 > 4 * kProjSteps)
          hot_gather<kProjSteps>(seq, e, lo, tb, Wb, x);
        if (t0 + 64 < n) {
          q.next(vals + a, cols + a, t0 + 64 * kProjQueue, n, mine);
          en = entry(t0 + 64);
        }
        hot_add<0>(seq, e.delta, w, acc);
        if (n - t0 > 4 * kProjSteps)
          hot_add<kProjSteps>(seq, e.delta, x, acc);
        e = en;
      }
      project_store<1>(acc, col_ok, grp, c4, D, cvec, E + row * lde);
      q = nq;
      a = na;
      n = nn;
    }
  }
}

}  // namespace sh

using namespace sh;

struct StatsPlan {
  int64_t n_chunks, spc, slab_rows;
};
static StatsPlan stats_plan(int64_t n_rows, int64_t chunk_rows) {
  StatsPlan p;
  if (chunk_rows <= 0 || chunk_rows > n_rows) chunk_rows = n_rows > 0 ? n_rows : 1;
  p.n_chunks = cdiv(n_rows > 0 ? n_rows : 1, chunk_rows);
  // one workgroup per slab: a whole number of fills of the GPU with about 256 rows each, so
  // that the last fill is not nearly empty; small matrices take smaller slabs, down to
  // kStatsMinRows rows (below that the accumulators' zeroing and writing outweigh them)
  const int64_t rows = std::max<int64_t>(n_rows, 1);
  const int64_t fills = std::max<int64_t>(1, (rows + 128 * kStatsResident) / (256 * kStatsResident));
  int64_t spc = fills * kStatsResident / p.n_chunks;
  if (10 * spc * p.n_chunks < 9 * fills * kStatsResident) ++spc;
  spc = std::max(spc, cdiv(chunk_rows, kStatsMaxRows));
  spc = std::max<int64_t>(1, std::min(spc, cdiv(chunk_rows, kStatsMinRows)));
  p.slab_rows = cdiv(chunk_rows, spc);
  p.spc = cdiv(chunk_rows, p.slab_rows);
  return p;
}

extern "C" size_t sh_norm_stats_workspace(int64_t n_rows, int64_t chunk_rows, int32_t d) {
  StatsPlan p = stats_plan(n_rows, chunk_rows);
  return (size_t)(p.n_chunks * p.spc) * 2 * (size_t)(d > 0 ? d : 1) * sizeof(double);
}

extern "C" int sh_norm_stats(const uint32_t *vals, const int32_t *cols, const int64_t *rowptr,
                             int64_t n_rows, int64_t chunk_rows, const int32_t *col_map,
                             int32_t n_cols_in, int32_t d, double sf, int log_transform,
                             const double *libsize_in, double *libsize_out, double *sum_out,
                             double *sumsq_out, void *workspace, size_t workspace_bytes,
                             sh_stream_t stream) {
  hipStream_t st = (hipStream_t)stream;
  SH_ARG(n_rows >= 0 && d > 0 && n_cols_in > 0, "sh_norm_stats: bad sizes n_rows=%lld d=%d n_cols_in=%d",
         (long long)n_rows, d, n_cols_in);
  SH_ARG(col_map || d == n_cols_in, "sh_norm_stats: col_map NULL requires d == n_cols_in");
  SH_ARG(rowptr && sum_out && sumsq_out, "sh_norm_stats: NULL pointer");
  SH_ARG(sf > 0, "sh_norm_stats: size factor must be > 0");
  if (n_rows == 0) {
    SH_HIP(hipMemsetAsync(sum_out, 0, sizeof(double) * d, st));
    SH_HIP(hipMemsetAsync(sumsq_out, 0, sizeof(double) * d, st));
    return SH_OK;
  }
  const StatsPlan plan = stats_plan(n_rows, chunk_rows);
  const int64_t chunk = (chunk_rows > 0 && chunk_rows < n_rows) ? chunk_rows : n_rows;
  const size_t need = sh_norm_stats_workspace(n_rows, chunk_rows, d);
  if (workspace_bytes < need || !workspace) {
    set_error("sh_norm_stats: workspace %zu < %zu bytes", workspace_bytes, need);
    return SH_EWORKSPACE;
  }
  const double *ls = libsize_in;
  if (!ls) {
    SH_ARG(libsize_out, "sh_norm_stats: libsize_out required when libsize_in is NULL");
    hipLaunchKernelGGL(k_libsize, dim3(cdiv(n_rows, 256 / kLibLanes)), dim3(256), 0, st, vals, cols, rowptr,
                       n_rows, col_map, n_cols_in, libsize_out);
    SH_LAUNCH_CHECK("k_libsize");
    ls = libsize_out;
  } else if (libsize_out && libsize_out != libsize_in) {
    SH_HIP(hipMemcpyAsync(libsize_out, libsize_in, sizeof(double) * n_rows,
                          hipMemcpyDeviceToDevice, st));
  }
  // accumulators of at most 2 x 2048 doubles (32 KiB) per workgroup: three on a CU; wider
  // matrices take column blocks (the CSR is re-read per block)
  const int32_t cb = d <= 2048 ? d : (int32_t)cdiv(d, cdiv(d, 2048));
  const int n_cb = (int)cdiv(d, cb);
  const size_t lds = (2 * (size_t)cb + 2 * (size_t)plan.slab_rows) * sizeof(double);
  double *part = (double *)workspace;
  hipLaunchKernelGGL(k_norm_stats, dim3((unsigned)(plan.n_chunks * plan.spc), n_cb),
                     dim3(kStatsThreads), lds, st, vals, cols, rowptr, n_rows, chunk,
                     (int)plan.spc, plan.slab_rows, col_map, n_cols_in, d, cb, sf, log_transform,
                     ls, part);
  SH_LAUNCH_CHECK("k_norm_stats");
  // chunks go in grid y (at most 65535 a launch)
  for (int64_t c0 = 0; c0 < plan.n_chunks; c0 += 65535) {
    const int64_t nc = std::min<int64_t>(65535, plan.n_chunks - c0);
    hipLaunchKernelGGL(k_reduce_slabs, dim3((unsigned)cdiv(d, kRedFeat), (unsigned)nc),
                       dim3(kRedFeat * kRedPart), 0, st,
                       part + (size_t)c0 * plan.spc * 2 * d, (int)plan.spc, d,
                       sum_out + c0 * d, sumsq_out + c0 * d);
  }
  SH_LAUNCH_CHECK("k_reduce_slabs");
  return SH_OK;
}

extern "C" int sh_stats_merge(const double *sums, const double *sumsqs, const int64_t *counts,
                              int32_t n_chunks, int32_t d, double *mu_out, double *sigma_out,
                              double *chunk_mean_out, sh_stream_t stream) {
  SH_ARG(n_chunks > 0 && d > 0, "sh_stats_merge: bad sizes");
  SH_ARG(sums && sumsqs && counts && mu_out && sigma_out, "sh_stats_merge: NULL pointer");
  hipLaunchKernelGGL(k_stats_merge, dim3(cdiv(d, 256)), dim3(256), 0, (hipStream_t)stream, sums,
                     sumsqs, counts, n_chunks, d, mu_out, sigma_out, chunk_mean_out);
  SH_LAUNCH_CHECK("k_stats_merge");
  return SH_OK;
}

extern "C" int sh_densify(const uint32_t *vals, const int32_t *cols, const int64_t *rowptr,
                          const int64_t *rows, int64_t n_rows, const int32_t *col_map,
                          int32_t n_cols_in, int32_t d, double sf, int log_transform,
                          const double *libsize, const double *center, const double *scale,
                          double clip, int out_f64, void *out, int64_t ld, sh_stream_t stream) {
  SH_ARG(n_rows >= 0 && d > 0 && ld >= d && ld % 4 == 0, "sh_densify: bad sizes d=%d ld=%lld", d,
         (long long)ld);
  SH_ARG(col_map || d == n_cols_in, "sh_densify: col_map NULL requires d == n_cols_in");
  SH_ARG(libsize && center && scale && out && rowptr, "sh_densify: NULL pointer");
  const size_t esz = out_f64 ? sizeof(double) : sizeof(float);
  SH_ARG(ld * esz <= 64 * 1024, "sh_densify: ld=%lld exceeds the 64 KiB row buffer",
         (long long)ld);
  if (n_rows == 0) return SH_OK;
  const int rpb = 2;
  if (out_f64)
    hipLaunchKernelGGL(k_densify<double>, dim3(cdiv(n_rows, rpb)), dim3(256), ld * esz,
                       (hipStream_t)stream, vals, cols, rowptr, rows, n_rows, col_map, n_cols_in,
                       d, sf, log_transform, libsize, center, scale, clip, (double *)out, ld, rpb);
  else
    hipLaunchKernelGGL(k_densify<float>, dim3(cdiv(n_rows, rpb)), dim3(256), ld * esz,
                       (hipStream_t)stream, vals, cols, rowptr, rows, n_rows, col_map, n_cols_in,
                       d, sf, log_transform, libsize, center, scale, clip, (float *)out, ld, rpb);
  SH_LAUNCH_CHECK("k_densify");
  return SH_OK;
}

extern "C" int sh_project(const uint32_t *vals, const int32_t *cols, const int64_t *rowptr,
                          int64_t n_rows, const int32_t *col_map, int32_t n_cols_in, int32_t d,
                          double sf, int log_transform, const double *libsize, const float *mu,
                          const float *inv_sigma, float clip, const float *W, int64_t ldw,
                          int32_t D, const float *c, float *E_out, int64_t lde,
                          sh_stream_t stream) {
  return sh_project_counted(vals, cols, rowptr, n_rows, -1, col_map, n_cols_in, d, sf,
                            log_transform, libsize, mu, inv_sigma, clip, W, ldw, D, c, E_out, lde,
                            stream);
}

extern "C" int sh_project_counted(const uint32_t *vals, const int32_t *cols,
                                  const int64_t *rowptr, int64_t n_rows, int64_t n_entries,
                                  const int32_t *col_map, int32_t n_cols_in, int32_t d, double sf,
                                  int log_transform, const double *libsize, const float *mu,
                                  const float *inv_sigma, float clip, const float *W, int64_t ldw,
                                  int32_t D, const float *c, float *E_out, int64_t lde,
                                  sh_stream_t stream) {
  SH_ARG(n_rows >= 0 && d > 0 && D > 0 && D <= 128 && ldw >= D && lde >= D,
         "sh_project: bad sizes d=%d D=%d ldw=%lld lde=%lld", d, D, (long long)ldw,
         (long long)lde);
  SH_ARG(col_map || d == n_cols_in, "sh_project: col_map NULL requires d == n_cols_in");
  SH_ARG(mu && inv_sigma && W && c && E_out && rowptr, "sh_project: NULL pointer");
  if (n_rows == 0) return SH_OK;
  SH_ARG(ldw % 4 == 0 && ((uintptr_t)W % 16) == 0,
         "sh_project: W rows must be 16-byte aligned (ldw a multiple of 4)");
  dim3 grid(cdiv(n_rows, 4)), block(256);
  // byte offsets into W in 32 bits, if it is that small
  const bool wide = (uint64_t)d * (uint64_t)ldw * 4 > 0xffffffffull;
  if (D <= 64 && n_rows >= kHotRows && d <= kHotMaxD && !wide &&
      (n_entries < 0 || hot_entries(n_rows, n_entries, libsize != nullptr))) {
    hipLaunchKernelGGL(col_map ? k_project_hot<true> : k_project_hot<false>, dim3(kHotBlocks),
                       dim3(kHotThreads), 0, (hipStream_t)stream, vals, cols, rowptr, n_rows,
                       col_map, n_cols_in, d, (float)sf, log_transform, libsize, mu, inv_sigma,
                       clip, W, ldw, D, c, E_out, lde);
    SH_LAUNCH_CHECK("k_project_hot");
    return SH_OK;
  }
  constexpr int kS = kProjSteps;
  auto kern = D <= 64                  ? (wide ? k_project<1, true, kS> : k_project<1, false, kS>)
              : n_rows <= kProjFewRows ? (wide ? k_project<2, true, kS> : k_project<2, false, kS>)
                                       : (wide ? k_project<2, true, kS / 2>
                                               : k_project<2, false, kS / 2>);
  hipLaunchKernelGGL(kern, grid, block, 0, (hipStream_t)stream, vals, cols, rowptr, n_rows,
                     col_map, n_cols_in, (float)sf, log_transform, libsize, mu, inv_sigma, clip, W,
                     ldw, D, c, E_out, lde);
  SH_LAUNCH_CHECK("k_project");
  return SH_OK;
}
