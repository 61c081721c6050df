// Fuzzy kNN edge weights: umap-learn's smooth_knn_dist + compute_membership_strengths
// as scarf applies them per row chunk (knn_utils.py:89-159), in float32 like the
// numba originals.
//
// Per chunk of `chunk_size` rows:
//   mean_c   = mean of all the chunk's distances (floor for rows with rho == 0)
//   rho_i    = local_connectivity-th non-zero distance (interpolated)
//   sigma_i  = bisection (<= n_iter steps) of sum_{j>=1} f(d_ij - rho_i) = log2(k) * bw,
//              f(x) = exp(-x / sigma) for x > 0 else 1, stop when |psum - target| < 1e-5;
//              floored at 1e-3 * mean(row) (rho > 0) or 1e-3 * mean_c
//   w_ij     = 0 if idx_ij equals the row's position inside the chunk, 1 if
//              d - rho <= 0 or sigma == 0, else exp(-(d - rho) / sigma)
// Then every zero weight becomes global_min: 1, lowered by each chunk that holds a
// zero weight to that chunk's smallest non-zero weight (knn_utils.py:144-158).
#include "sh_common.h"

namespace sh {

constexpr float kSmoothTol = 1e-5f;
constexpr float kMinKDistScale = 1e-3f;

// Deterministic FP64 mean of each chunk's n_c * k distances.  A chunk's entries are cut
// into mean_parts(chunk_size) contiguous parts, one workgroup each (20 chunks at 1M rows
// would otherwise leave the GPU nearly idle); each part sums in a fixed tree order and the
// parts are added in order, so the result depends only on the inputs.
constexpr int kMeanParts = 64;
inline int64_t mean_parts(int64_t cs) { return std::min<int64_t>(kMeanParts, cdiv(cs, 128)); }

__global__ void __launch_bounds__(256) k_chunk_mean_part(const float *__restrict__ dist,
                                                         int64_t n, int32_t k, int64_t cs,
                                                         int32_t parts,
                                                         double *__restrict__ part_out) {
  __shared__ double red[256];
  const int64_t c = blockIdx.x;
  const int64_t a = c * cs * k, b = min(n, (c + 1) * cs) * (int64_t)k;
  const int64_t len = (b - a + parts - 1) / parts;
  const int64_t pa = min(b, a + (int64_t)blockIdx.y * len), pb = min(b, pa + len);
  double s = 0.0;
  for (int64_t t = pa + threadIdx.x; t < pb; t += 256) s += (double)dist[t];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part_out[c * parts + blockIdx.y] = red[0];
}

__global__ void __launch_bounds__(256) k_chunk_mean_sum(const double *__restrict__ part,
                                                        int64_t n, int32_t k, int64_t cs,
                                                        int32_t parts, int64_t nc,
                                                        double *__restrict__ mean_out) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const int64_t cnt = (min(n, (c + 1) * cs) - c * cs) * (int64_t)k;
  double s = 0.0;
  for (int p = 0; p < parts; ++p) s += part[c * parts + p];
  mean_out[c] = cnt > 0 ? s / (double)cnt : 0.0;
}

// rho of one row: the local_connectivity-th non-zero distance (interpolated).  d holds zeros
// past the row's k distances.
template <int KM>
__device__ __forceinline__ float smooth_rho(const float (&d)[KM], float lc) {
  int nnz = 0;
#pragma unroll
  for (int j = 0; j < KM; ++j)
    if (d[j] > 0.f) ++nnz;
  float rho = 0.f;
  if ((float)nnz >= lc) {
    const int index = (int)floorf(lc);
    const float interp = lc - (float)index;
    float nz_prev = 0.f, nz_at = 0.f;  // non-zero distances index-1 and index
    int seen = 0;
#pragma unroll
    for (int j = 0; j < KM; ++j) {
      if (d[j] > 0.f) {
        if (seen == index - 1) nz_prev = d[j];
        if (seen == index) nz_at = d[j];
        ++seen;
      }
    }
    if (index > 0) {
      rho = nz_prev;
      if (interp > kSmoothTol) rho += interp * (nz_at - nz_prev);
    } else {
      float first = 0.f;
      bool got = false;
#pragma unroll
      for (int j = 0; j < KM; ++j)
        if (!got && d[j] > 0.f) {
          first = d[j];
          got = true;
        }
      rho = interp * first;
    }
  } else if (nnz > 0) {
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < KM; ++j)
      if (d[j] > 0.f) mx = fmaxf(mx, d[j]);
    rho = mx;
  }
  return rho;
}

// sigma of one row by umap's bisection, with the evaluations that cannot matter left out.
// The sum is monotone in sigma, so far from its root only the sign of mid - root decides a
// step, and neither the stop test nor a rounding can come into it.  A few safeguarded Newton
// steps (hardware exp and reciprocal) place the root to about 1e-7; within 5e-5 / slope of
// it, five times the stop tolerance, a step evaluates the sum as before, so every midpoint,
// and the sigma, is the one that the plain bisection gives.  Where Newton does not settle
// (a flat sum, non-finite distances) every step evaluates.  gap[j] = d[j] - rho,
// infinite past the row's k distances: no test of j < k (their masks did not fit the scalar
// registers), and a term of exactly zero.
template <int KM>
__device__ __forceinline__ float smooth_sigma(const float (&gap)[KM], int32_t k, double target,
                                              int32_t n_iter) {
  float root = 0.f, near = INFINITY;
  // Rows without a root decide the same way at every step: 64 evaluations of each, with the
  // padded terms, took 1M rows of 2 from 0.21 to 0.51 ms.  0.01 is far more than the sums'
  // rounding and the tolerance.
  const float t = (float)target;
  if ((float)(k - 1) < t - 0.01f) {  // the sum is below the target
    root = INFINITY;
    near = 0.f;
  } else {
    float gaps = 0.f;
#pragma unroll
    for (int j = 1; j < KM; ++j) gaps += gap[j] < INFINITY ? fmaxf(gap[j], 0.f) : 0.f;
    float x = gaps / (float)(k > 1 ? k - 1 : 1);
    for (int it = 0; it < 14; ++it) {
      const float inv = __builtin_amdgcn_rcpf(x) * -1.44269504f;  // exp2 argument per gap
      float f = -t, s = 0.f;  // sum - target, and x times its derivative
#pragma unroll
      for (int j = 1; j < KM; ++j) {
        const float a = fmaxf(fmaxf(gap[j], 0.f) * inv, -256.f);  // exp2(-256) is 0
        const float e = __builtin_amdgcn_exp2f(a);
        f += e;
        s = fmaf(-a, e, s);
      }
      s *= 0.693147181f;
      if (!(s > 1e-2f && x < 1e30f && x > 1e-30f)) break;
      const float step = fminf(fmaxf(-f / s, -2.f), 2.f);
      if (fabsf(f) < 2e-6f * (float)k) {
        root = x * (1.f + step);
        near = root * (5e-5f / s);
        break;
      }
      x *= __builtin_amdgcn_exp2f(step * 1.44269504f);
    }
    if (near == INFINITY) {
      int ones = 0, less = 0;  // terms of 1 whatever sigma, and of less than that
#pragma unroll
      for (int j = 1; j < KM; ++j) {
        ones += !(gap[j] > 0.f);
        less += gap[j] > 0.f && gap[j] < INFINITY;
      }
      if ((float)ones > t + 0.01f) {
        root = -1.f;
        near = 0.f;
      } else if ((float)(ones + less) < t - 0.01f) {
        root = INFINITY;
        near = 0.f;
      }
    }
  }
  float lo = 0.f, hi = INFINITY, mid = 1.f;
  for (int it = 0; it < n_iter; ++it) {
    bool above;
    if (fabsf(mid - root) > near) {
      above = mid > root;
    } else {
      float psum = 0.f;
#pragma unroll
      for (int j = 1; j < KM; ++j)
        psum = gap[j] > 0.f ? psum + expf(-(gap[j] / mid)) : psum + 1.f;
      if (fabs((double)psum - target) < (double)kSmoothTol) break;
      above = (double)psum > target;
    }
    if (above) {
      hi = mid;
      mid = (lo + hi) / 2.f;
    } else {
      lo = mid;
      if (hi == INFINITY)
        mid = mid * 2.f;
      else
        mid = (lo + hi) / 2.f;
    }
  }
  return mid;
}

// One thread per row for rho and sigma, then the workgroup's weights element by element.  The
// distances come in and the weights go out coalesced (a thread walking its own row touched
// a line per lane); the rows in between pass through LDS.
// 1M x 21: 453 -> 300 us.
template <int KM>
__global__ void __launch_bounds__(256) k_smooth_rows(
    const float *__restrict__ dist, const int64_t *__restrict__ idx, int64_t n, int32_t k,
    int64_t cs, float lc, float bw, int32_t n_iter, const double *__restrict__ chunk_mean,
    float *__restrict__ sigma_out, float *__restrict__ rho_out, float *__restrict__ w_out,
    uint32_t *__restrict__ chunk_minw, int32_t *__restrict__ chunk_zero,
    uint8_t *__restrict__ block_zero) {
  extern __shared__ float sd[];  // [256][k | 1]
  __shared__ float s_rho[256], s_sigma[256];
  __shared__ int any_zero_block;
  __shared__ uint32_t s_min[256];  // per row, where the workgroup's rows span chunks
  __shared__ int s_zero[256];
  const int ld = k | 1;
  const int64_t r0 = (int64_t)blockIdx.x * 256;
  const int rows = (int)min<int64_t>(256, n - r0);
  const int tid = threadIdx.x;
  const int total = rows * k;
  for (int e = tid; e < total; e += 256) sd[(e / k) * ld + e % k] = dist[r0 * k + e];
  if (tid == 0) any_zero_block = 0;
  s_min[tid] = 0xffffffffu;
  s_zero[tid] = 0;
  __syncthreads();
  if (tid < rows) {
    const int64_t i = r0 + tid;
    float d[KM];
    double rs = 0.0;
#pragma unroll
    for (int j = 0; j < KM; ++j) {
      d[j] = j < k ? sd[tid * ld + j] : 0.f;
      rs += (double)d[j];
    }
    const float row_mean = (float)(rs / (double)k);
    const float mean_c = (float)chunk_mean[i / cs];
    const float rho = smooth_rho<KM>(d, lc);
#pragma unroll
    for (int j = 0; j < KM; ++j) d[j] = j < k ? d[j] - rho : INFINITY;
    float sigma = smooth_sigma<KM>(d, k, log2((double)k) * (double)bw, n_iter);
    if (rho > 0.f) {
      if (sigma < kMinKDistScale * row_mean) sigma = kMinKDistScale * row_mean;
    } else {
      if (sigma < kMinKDistScale * mean_c) sigma = kMinKDistScale * mean_c;
    }
    sigma_out[i] = sigma;
    rho_out[i] = rho;
    s_rho[tid] = rho;
    s_sigma[tid] = sigma;
  }
  __syncthreads();
  // Chunk minimum and zero flag: registers, then one atomic per wave and quantity where the
  // workgroup's rows share a chunk; else per row in LDS and then per wave or row (thousands
  // of global atomics of one workgroup on the same two words took 0.9 ms).  Neither depends
  // on order.
  const int64_t c0 = r0 / cs;
  const bool one_chunk = (r0 + rows - 1) / cs == c0;
  uint32_t minw = 0xffffffffu;
  int zero = 0;
  for (int e = tid; e < total; e += 256) {
    const int r = e / k;
    const int64_t i = r0 + r;
    const int64_t local = one_chunk ? i - c0 * cs : i % cs;
    const float dd = sd[r * ld + e % k] - s_rho[r];
    float w;
    if (idx[r0 * k + e] == local)
      w = 0.f;
    else if (dd <= 0.f || s_sigma[r] == 0.f)
      w = 1.f;
    else
      w = expf(-(dd / s_sigma[r]));
    w_out[r0 * k + e] = w;
    if (w == 0.f) {
      zero = 1;
      if (!one_chunk) s_zero[r] = 1;
    } else {
      minw = min(minw, float_ord(w));
      if (!one_chunk) atomicMin(&s_min[r], float_ord(w));
    }
  }
  if (__ballot(zero) != 0 && (tid & 63) == 0) any_zero_block = 1;
  __syncthreads();
  if (tid == 0) block_zero[blockIdx.x] = (uint8_t)any_zero_block;
  int64_t c = c0;
  if (!one_chunk) {  // this thread's row
    if (tid >= rows) return;
    c = (r0 + tid) / cs;
    minw = s_min[tid];
    zero = s_zero[tid];
  }
  if (__ballot(1) == ~0ull && __ballot(c != __shfl(c, 0, 64)) == 0) {
    const bool any_zero = __ballot(zero) != 0;
    for (int o = 32; o >= 1; o >>= 1) minw = min(minw, (uint32_t)__shfl_xor((int)minw, o, 64));
    if ((tid & 63) == 0) {
      if (any_zero) atomicOr(&chunk_zero[c], 1);
      if (minw != 0xffffffffu) atomicMin(&chunk_minw[c], minw);
    }
  } else {
    if (zero) atomicOr(&chunk_zero[c], 1);
    if (minw != 0xffffffffu) atomicMin(&chunk_minw[c], minw);
  }
}

// global_min over the chunks that hold a zero weight (one workgroup; a minimum does not
// depend on order).
__global__ void __launch_bounds__(256) k_global_min(const uint32_t *__restrict__ chunk_minw,
                                                    const int32_t *__restrict__ chunk_zero,
                                                    int64_t n_chunks, float *__restrict__ gmin) {
  __shared__ float red[4];
  float g = 1.f;
  for (int64_t c = threadIdx.x; c < n_chunks; c += 256)
    if (chunk_zero[c] && chunk_minw[c] != 0xffffffffu) {
      const float m = ord_float(chunk_minw[c]);
      if (m < g) g = m;
    }
  for (int o = 32; o >= 1; o >>= 1) g = fminf(g, __shfl_xor(g, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = g;
  __syncthreads();
  if (threadIdx.x == 0) *gmin = fminf(fminf(red[0], red[1]), fminf(red[2], red[3]));
}

// Only the blocks that wrote a zero are read again.
__global__ void __launch_bounds__(256) k_fix_zero(float *__restrict__ w, int64_t n, int32_t k,
                                                  const uint8_t *__restrict__ block_zero,
                                                  const float *__restrict__ gmin) {
  if (!block_zero[blockIdx.x]) return;
  const int64_t r0 = (int64_t)blockIdx.x * 256;
  const int total = (int)min<int64_t>(256, n - r0) * k;
  for (int e = threadIdx.x; e < total; e += 256)
    if (w[r0 * k + e] == 0.f) w[r0 * k + e] = *gmin;
}

__global__ void k_smooth_init(uint32_t *__restrict__ chunk_minw, int32_t *__restrict__ chunk_zero,
                              int64_t n_chunks) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n_chunks) {
    chunk_minw[t] = 0xffffffffu;
    chunk_zero[t] = 0;
  }
}

}  // namespace sh

using namespace sh;

extern "C" size_t sh_smooth_knn_workspace(int64_t n, int64_t chunk_size) {
  if (chunk_size <= 0) return 0;
  const int64_t nc = cdiv(n, chunk_size);
  return align_up(nc * sizeof(double), 256) + align_up(nc * sizeof(uint32_t), 256) +
         align_up(nc * sizeof(int32_t), 256) + 256 +
         align_up(nc * mean_parts(chunk_size) * sizeof(double), 256) +
         align_up((size_t)cdiv(n, 256), 256);
}

extern "C" int sh_smooth_knn(const float *dist, const int64_t *idx, int64_t n, int32_t k,
                             int64_t chunk_size, float local_connectivity, float bandwidth,
                             int32_t n_iter, float *sigma_out, float *rho_out, float *w_out,
                             void *workspace, size_t workspace_bytes, sh_stream_t stream) {
  SH_ARG(n >= 0 && k >= 1 && k <= 64, "sh_smooth_knn: k=%d must be in [1, 64]", k);
  SH_ARG(chunk_size >= 1, "sh_smooth_knn: chunk_size must be >= 1");
  SH_ARG(dist && idx && sigma_out && rho_out && w_out, "sh_smooth_knn: NULL pointer");
  if (n == 0) return SH_OK;
  const size_t need = sh_smooth_knn_workspace(n, chunk_size);
  if (!workspace || workspace_bytes < need) {
    set_error("sh_smooth_knn: workspace %zu < %zu bytes", workspace_bytes, need);
    return SH_EWORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nc = cdiv(n, chunk_size);
  char *p = (char *)workspace;
  double *cmean = (double *)p;
  p += align_up(nc * sizeof(double), 256);
  uint32_t *cmin = (uint32_t *)p;
  p += align_up(nc * sizeof(uint32_t), 256);
  int32_t *czero = (int32_t *)p;
  p += align_up(nc * sizeof(int32_t), 256);
  float *gmin = (float *)p;
  p += 256;
  double *cpart = (double *)p;
  p += align_up(nc * mean_parts(chunk_size) * sizeof(double), 256);
  uint8_t *bzero = (uint8_t *)p;
  hipLaunchKernelGGL(k_smooth_init, dim3(cdiv(nc, 256)), dim3(256), 0, st, cmin, czero, nc);
  SH_LAUNCH_CHECK("k_smooth_init");
  const int32_t parts = (int32_t)mean_parts(chunk_size);
  hipLaunchKernelGGL(k_chunk_mean_part, dim3(nc, parts), dim3(256), 0, st, dist, n, k,
                     chunk_size, parts, cpart);
  SH_LAUNCH_CHECK("k_chunk_mean_part");
  hipLaunchKernelGGL(k_chunk_mean_sum, dim3(cdiv(nc, 256)), dim3(256), 0, st, cpart, n, k,
                     chunk_size, parts, nc, cmean);
  SH_LAUNCH_CHECK("k_chunk_mean_sum");
  dim3 grid(cdiv(n, 256)), block(256);
  const size_t lds = 256 * (size_t)(k | 1) * sizeof(float);  // at most 65 KB of a CU's 160
#define SH_SMOOTH(KM)                                                                           \
  hipLaunchKernelGGL(k_smooth_rows<KM>, grid, block, lds, st, dist, idx, n, k, chunk_size,      \
                     local_connectivity, bandwidth, n_iter, cmean, sigma_out, rho_out, w_out,   \
                     cmin, czero, bzero)
  if (k <= 12)
    SH_SMOOTH(12);
  else if (k <= 16)
    SH_SMOOTH(16);
  else if (k <= 24)
    SH_SMOOTH(24);
  else if (k <= 32)
    SH_SMOOTH(32);
  else if (k <= 48)
    SH_SMOOTH(48);
  else
    SH_SMOOTH(64);
#undef SH_SMOOTH
  SH_LAUNCH_CHECK("k_smooth_rows");
  hipLaunchKernelGGL(k_global_min, dim3(1), dim3(256), 0, st, cmin, czero, nc, gmin);
  SH_LAUNCH_CHECK("k_global_min");
  hipLaunchKernelGGL(k_fix_zero, grid, block, 0, st, w_out, n, k, bzero, gmin);
  SH_LAUNCH_CHECK("k_fix_zero");
  return SH_OK;
}
