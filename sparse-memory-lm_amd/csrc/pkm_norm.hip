// 2-norm of a value table's gradient accumulator (clip_row_sparse, smlm/sparse_values.py) over the rows that a backward
// flagged; every other row of the accumulator is zero.
//
// Bound by the flagged rows' bytes.  A norm over the whole accumulator reads all of it: 1,048,576 x 384 fp32 with 40%
// of the rows flagged 426 us, 8,388,592 x 24 with 0.6% 215 us; here 156 and 17 us (with the second
// launch 159 and 20).  Widths that are no multiple of 4 are read column by column: 1,000,000 x 385 with 5 / 40 / 100% of the
// rows flagged 46 / 255 / 497 us, 383 for the norm of the whole (16 loads in flight 490, a row at a time 443 at 100%).
#include "pkm_common.h"

namespace smlm {
namespace {

constexpr int kNormThreads = 256;
constexpr int kNormWaves = kNormThreads / kWave;
constexpr int kNormScan = 256;    // most flags that a wavefront reads at a time
constexpr int kNormParts = 2048;  // workgroups of the first launch: 8 wavefronts per SIMD

__device__ __forceinline__ double wave_sum_f64(double v) {
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__device__ __forceinline__ double block_sum_f64(double v) {
  __shared__ double s[kNormWaves];
  v = wave_sum_f64(v);
  if (lane_id() == 0) s[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kNormWaves; ++w) t += s[w];
  return t;
}

// A wavefront lists the flagged rows among `scan` in LDS and sums the squares of their columns, V per lane at a time,
// the lanes running through the listed rows as if they were one; squares and sums in 64 bits.
template <int V>
__global__ void __launch_bounds__(kNormThreads)
    flagged_squares_kernel(const float *__restrict__ acc, const uint8_t *__restrict__ touched, int64_t rows, int D,
                           int scan, double *__restrict__ parts) {
  __shared__ uint16_t lists[kNormWaves][kNormScan];
  uint16_t *list = lists[threadIdx.x / kWave];
  const int lane = lane_id();
  const int per_row = D / V, row_step = kWave / per_row, col_step = kWave % per_row;  // D % V == 0
  double sum = 0.0;
  for (int64_t row0 = ((int64_t)blockIdx.x * kNormWaves + threadIdx.x / kWave) * scan; row0 < rows;
       row0 += (int64_t)gridDim.x * kNormWaves * scan) {
    int count = 0;
#pragma unroll
    for (int i = 0; i < kNormScan; i += kWave) {
      if (i >= scan) break;
      const int64_t r = row0 + i + lane;
      const bool flag = i + lane < scan && r < rows && touched[r] != 0;
      const uint64_t mask = ballot(flag);
      if (flag) list[count + lanes_below(mask)] = (uint16_t)(i + lane);
      count += __popcll(mask);
    }
    wave_lds_sync();
    int k = lane / per_row, c = lane % per_row;  // this lane's row of the list and chunk of the row
    while (k < count) {
      float x[4][V];
#pragma unroll
      for (int u = 0; u < 4; ++u) {              // four loads in flight; past the list's end they add nothing
        const bool live = k < count;
        const float *src = acc + (row0 + list[live ? k : 0]) * D + c * V;
        if constexpr (V == 4) {
          const float4 t = *(const float4 *)src;
          x[u][0] = live ? t.x : 0.f, x[u][1] = live ? t.y : 0.f, x[u][2] = live ? t.z : 0.f, x[u][3] = live ? t.w : 0.f;
        } else {
          x[u][0] = live ? src[0] : 0.f;
        }
        k += row_step;
        c += col_step;
        if (c >= per_row) { c -= per_row; ++k; }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < V; ++e) sum = __builtin_fma((double)x[u][e], (double)x[u][e], sum);
    }
    wave_lds_sync();  // the list is rewritten by the next scan
  }
  sum = block_sum_f64(sum);
  if (threadIdx.x == 0) parts[blockIdx.x] = sum;
}

// The parts in a fixed order; the sum is rounded to fp32 before the root, so that it overflows where an fp32 sum does.
// out[1]: the clip factor min(1, max_norm / (norm + 1e-6)) as torch evaluates it (a NaN stays one).
__global__ void __launch_bounds__(kNormThreads)
    norm_of_parts_kernel(const double *__restrict__ parts, int n, float max_norm, float *__restrict__ out) {
  double sum = 0.0;
  for (int i = threadIdx.x; i < n; i += kNormThreads) sum += parts[i];
  sum = block_sum_f64(sum);
  if (threadIdx.x != 0) return;
  const float norm = sqrtf((float)sum), factor = 1.0f / (norm + 1e-6f) * max_norm;
  out[0] = norm;
  out[1] = factor > 1.0f ? 1.0f : factor;
}

}  // namespace
}  // namespace smlm

extern "C" int smlm_flagged_norm_parts(void) { return smlm::kNormParts; }

extern "C" int smlm_flagged_norm(const float *acc, const uint8_t *touched, int64_t rows, int D, float max_norm,
                                 double *parts, float *out, void *stream) {
  using namespace smlm;
  if (!acc || !touched || !parts || !out) return fail(SMLM_EINVAL, "smlm_flagged_norm: null pointer argument");
  if (rows < 0 || D < 1) return fail(SMLM_EINVAL, "smlm_flagged_norm: bad shape rows=%lld D=%d", (long long)rows, D);
  // 256 flags at a time where that leaves every wavefront of the launch a scan, else 64
  const int scan = rows / kNormScan >= kNormParts * kNormWaves / 2 ? kNormScan : kWave;
  const int64_t scans = (rows + scan - 1) / scan, want = (scans + kNormWaves - 1) / kNormWaves;
  const int blocks = (int)(want < 1 ? 1 : want > kNormParts ? kNormParts : want);
  hipStream_t s = (hipStream_t)stream;
  if (D % 4 == 0 && (uintptr_t)acc % 16 == 0)
    hipLaunchKernelGGL((flagged_squares_kernel<4>), dim3(blocks), dim3(kNormThreads), 0, s, acc, touched, rows, D, scan,
                       parts);
  else
    hipLaunchKernelGGL((flagged_squares_kernel<1>), dim3(blocks), dim3(kNormThreads), 0, s, acc, touched, rows, D, scan,
                       parts);
  hipLaunchKernelGGL(norm_of_parts_kernel, dim3(1), dim3(kNormThreads), 0, s, parts, blocks, max_norm, out);
  return launch_status("smlm_flagged_norm");
}
