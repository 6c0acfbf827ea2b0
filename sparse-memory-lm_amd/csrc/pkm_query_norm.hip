// Gradient of the memory query's batch normalisation in training (smlm/pkm.py:188-191): from the bf16 projection x and
// the gradient g of the bf16 result, with the fp32 statistics of the forward.
//
// Bound by reading x and g twice and writing dx once (4,096 x 2,048: 84 MB in bf16).  torch's gradient on fp32 copies took
// 200 us there (cast 9, column reductions 160, elements 17, cast back 9, fill 4): its reductions keep few wavefronts
// busy.  Here the sums run over (row chunk, 256 columns) workgroups, 16 bytes per lane: 30 us.  Sums in 64 bits,
// in a fixed order.  (The forward stays torch's: statistics that differ in their last bit move some of the rounded
// queries, and with them selections.)
#include <algorithm>

#include "pkm_common.h"

namespace smlm {
namespace {

constexpr int kQnThreads = 256;
constexpr int kQnCols = 256;                   // columns per workgroup: 32 lanes x 8
constexpr int kQnRows = kQnThreads / 32;       // rows a workgroup reads at a time
constexpr int kQnChunks = 128;                 // most row chunks

__device__ __forceinline__ void unpack8(const uint4 v, float *x) {
  const uint32_t t[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) x[2 * i] = __uint_as_float(t[i] << 16), x[2 * i + 1] = __uint_as_float(t[i] & 0xFFFF0000u);
}

// Column sums of one chunk of rows: of g and of g (x - mean).
__global__ void __launch_bounds__(kQnThreads)
    query_norm_sums_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ g, const float *__restrict__ mean,
                           int64_t N, int C, int64_t rows_per_chunk, double *__restrict__ parts) {
  __shared__ double s[kQnRows][2][kQnCols];
  const int sub = threadIdx.x % 32, rl = threadIdx.x / 32, col = blockIdx.x * kQnCols + sub * 8;
  const int64_t r0 = blockIdx.y * rows_per_chunk, r1 = min(N, r0 + rows_per_chunk);
  double a[8] = {}, b[8] = {};
  if (col < C) {                               // C % 8 == 0
    float mu[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) mu[e] = mean[col + e];
#pragma unroll 4
    for (int64_t r = r0 + rl; r < r1; r += kQnRows) {
      float v[8], w[8];
      unpack8(*(const uint4 *)(x + r * C + col), v);
      unpack8(*(const uint4 *)(g + r * C + col), w);
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] += w[e], b[e] += (double)(w[e] * (v[e] - mu[e]));
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s[rl][0][sub * 8 + e] = a[e], s[rl][1][sub * 8 + e] = b[e];
  __syncthreads();
  const int c = blockIdx.x * kQnCols + threadIdx.x;
  if (c >= C) return;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    double sum = 0.0;
    for (int r = 0; r < kQnRows; ++r) sum += s[r][k][threadIdx.x];
    parts[((int64_t)blockIdx.y * 2 + k) * C + c] = sum;
  }
}

// dweight and dbias, and the two columns of factors of the gradient: dx = (g - k0 - (x - mean) k1) invstd w.
__global__ void __launch_bounds__(kQnThreads)
    query_norm_columns_kernel(const double *__restrict__ parts, int chunks, int64_t N, int C,
                              const float *__restrict__ invstd, float *__restrict__ dweight, float *__restrict__ dbias,
                              float *__restrict__ k) {
  const int c = blockIdx.x * kQnThreads + threadIdx.x;
  if (c >= C) return;
  double a = 0.0, b = 0.0;
#pragma unroll 8
  for (int i = 0; i < chunks; ++i) {
    a += parts[(int64_t)(2 * i) * C + c];
    b += parts[(int64_t)(2 * i + 1) * C + c];
  }
  const double is = invstd[c];
  dbias[c] = (float)a;
  dweight[c] = (float)(b * is);
  k[c] = (float)(a / (double)N);
  k[C + c] = (float)(b * is * is / (double)N);
}

__global__ void __launch_bounds__(kQnThreads)
    query_norm_rows_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ g, const float *__restrict__ mean,
                           const float *__restrict__ invstd, const float *__restrict__ weight,
                           const float *__restrict__ k, int64_t vecs, int cols8, int C, uint16_t *__restrict__ dx) {
  for (int64_t i = (int64_t)blockIdx.x * kQnThreads + threadIdx.x; i < vecs; i += (int64_t)gridDim.x * kQnThreads) {
    const int col = (int)(i % cols8) * 8;
    float v[8], w[8];
    unpack8(*(const uint4 *)(x + i * 8), v);
    unpack8(*(const uint4 *)(g + i * 8), w);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int c = col + e;
      v[e] = (w[e] - k[c] - (v[e] - mean[c]) * k[C + c]) * (invstd[c] * weight[c]);
    }
    *(uint4 *)(dx + i * 8) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                                        pack_bf16x2(v[6], v[7]));
  }
}

struct QnShape {
  int chunks, col_blocks, cols8;
  int64_t rows_per_chunk, vecs;
  unsigned row_grid;
};
QnShape qn_shape(int64_t N, int C) {
  QnShape s;
  s.col_blocks = (C + kQnCols - 1) / kQnCols;
  // two workgroups per CU if the rows allow it, at least 32 rows each
  const int64_t want = std::max<int64_t>(1, std::min<int64_t>(kQnChunks, 512 / s.col_blocks));
  s.rows_per_chunk = std::max<int64_t>(32, (N + want - 1) / want);
  s.chunks = (int)((N + s.rows_per_chunk - 1) / s.rows_per_chunk);
  s.cols8 = C / 8;
  s.vecs = N * s.cols8;
  s.row_grid = (unsigned)std::min<int64_t>((s.vecs + kQnThreads - 1) / kQnThreads, 1 << 16);
  return s;
}

}  // namespace
}  // namespace smlm

extern "C" int64_t smlm_query_norm_parts(int64_t N, int C) {
  return N < 1 || C < 1 ? 0 : (int64_t)smlm::qn_shape(N, C).chunks * 2 * C;
}

extern "C" int smlm_query_norm_backward(const void *g, const void *x, const float *weight, const float *mean,
                                        const float *invstd, int64_t N, int C, double *parts, float *k, void *dx,
                                        float *dweight, float *dbias, void *stream) {
  using namespace smlm;
  const void *const p16[] = {g, x, dx, parts};
  for (const void *p : p16)
    if (!p || (uintptr_t)p % 16)
      return fail(SMLM_EINVAL, "smlm_query_norm_backward: g, x, dx and parts must be 16-byte aligned, not null");
  if (!weight || !mean || !invstd || !k || !dweight || !dbias)
    return fail(SMLM_EINVAL, "smlm_query_norm_backward: null pointer argument");
  if (N < 2 || N > (int64_t)1 << 40 || C < 8 || C % 8 || C > (1 << 20))
    return fail(SMLM_EUNSUPPORTED, "smlm_query_norm_backward: N=%lld C=%d (at least two rows, C a multiple of 8)",
                (long long)N, C);
  const QnShape q = qn_shape(N, C);
  hipStream_t s = (hipStream_t)stream;
  const dim3 block(kQnThreads);
  hipLaunchKernelGGL(query_norm_sums_kernel, dim3(q.col_blocks, q.chunks), block, 0, s, (const uint16_t *)x,
                     (const uint16_t *)g, mean, N, C, q.rows_per_chunk, parts);
  hipLaunchKernelGGL(query_norm_columns_kernel, dim3((unsigned)((C + kQnThreads - 1) / kQnThreads)), block, 0, s, parts,
                     q.chunks, N, C, invstd, dweight, dbias, k);
  hipLaunchKernelGGL(query_norm_rows_kernel, dim3(q.row_grid), block, 0, s, (const uint16_t *)x, (const uint16_t *)g,
                     mean, invstd, weight, k, q.vecs, q.cols8, C, (uint16_t *)dx);
  return launch_status("smlm_query_norm_backward");
}
