// Row quantisation of the value table for the inference bag (int8 and packed 4-bit, one fp16 scale per row).
// The scheme is the one of scripts/quantize_table_eval.py:45-61 (int8) and smlm/kernels.py:280-300 (q4):
//   m    = the row's value of largest magnitude (the first one on ties, as torch.argmax)
//   d    = fp16(m / lo), replaced by 1 if it is zero
//   code = clamp(round_half_even(w / d), lo, hi)            (fp32 division, correctly rounded)
// int8: (lo, hi) = (-128, 127), codes stored as int8.  q4: (lo, hi) = (-8, 7), byte i of a row holds column i
// in the low nibble and column i + D/2 in the high nibble, each as code + 8.
// Two layouts: quantize_rows_kernel (16 lanes per row, the row in registers) for widths of whole 16-byte chunks, and
// quantize_kernel (one wavefront per row, four rows per workgroup) for every other width or alignment.
#include "pkm_common.h"

namespace smlm {
namespace {

template <bool SRC_F32>
__device__ __forceinline__ float src_val(const void *src, int64_t o) {
  if constexpr (SRC_F32) return ((const float *)src)[o];
  else return bf16_bits_to_f32(((const uint16_t *)src)[o]);
}

template <bool SRC_F32, bool Q4>
__global__ void __launch_bounds__(256) quantize_kernel(const void *__restrict__ src, int64_t rows, int D,
                                                       void *__restrict__ codes, uint16_t *__restrict__ scales) {
  const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
  if (row >= rows) return;
  const int lane = lane_id();
  const int64_t base = row * D;

  float best = -1.f;
  int bi = 0x7FFFFFFF;
  for (int col = lane; col < D; col += kWave) {
    const float a = fabsf(src_val<SRC_F32>(src, base + col));
    if (a > best) { best = a; bi = col; }
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, kWave);
    const int oi = __shfl_xor(bi, o, kWave);
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
  }
  if (bi >= D) bi = 0;  // a row without any ordered value (all NaN) still reads in bounds
  const float lo = Q4 ? -8.f : -128.f, hi = Q4 ? 7.f : 127.f;
  const float m = src_val<SRC_F32>(src, base + bi);
  uint16_t db = f32_to_f16_bits(m / lo);
  if ((db & 0x7FFFu) == 0) db = 0x3C00u;  // fp16 1.0
  const float d = f16_bits_to_f32(db);
  if (lane == 0) scales[row] = db;

  if constexpr (!Q4) {
    int8_t *out = (int8_t *)codes + base;
    for (int col = lane; col < D; col += kWave)
      out[col] = (int8_t)fminf(fmaxf(rintf(src_val<SRC_F32>(src, base + col) / d), lo), hi);
  } else {
    const int half = D / 2;
    uint8_t *out = (uint8_t *)codes + row * half;
    for (int col = lane; col < half; col += kWave) {
      const int c0 = (int)fminf(fmaxf(rintf(src_val<SRC_F32>(src, base + col) / d), lo), hi) + 8;
      const int c1 = (int)fminf(fmaxf(rintf(src_val<SRC_F32>(src, base + half + col) / d), lo), hi) + 8;
      out[col] = (uint8_t)(c0 | (c1 << 4));
    }
  }
}

// Four values of a row, at a multiple of four columns.
template <bool SRC_F32>
__device__ __forceinline__ void load4(const void *src, int64_t o, float *x) {
  if constexpr (SRC_F32) {
    const float4 t = *(const float4 *)((const float *)src + o);
    x[0] = t.x, x[1] = t.y, x[2] = t.z, x[3] = t.w;
  } else {
    const uint2 t = *(const uint2 *)((const uint16_t *)src + o);
    x[0] = bf16_bits_to_f32(t.x & 0xFFFFu), x[1] = bf16_bits_to_f32(t.x >> 16);
    x[2] = bf16_bits_to_f32(t.y & 0xFFFFu), x[3] = bf16_bits_to_f32(t.y >> 16);
  }
}

// The larger of (best, bi) and lane ^ J's pair: the greater magnitude, the lower column of equal ones.
template <int J>
__device__ __forceinline__ void argmax_step(float &best, int &bi) {
  const float ob = __uint_as_float(xor_lane<J>(__float_as_uint(best)));
  const int oi = (int)xor_lane<J>((uint32_t)bi);
  if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
}

// Bound by the row's read (1,536 bytes of fp32 for 384 codes).  quantize_kernel reads 4 bytes per lane, reads every
// row twice, reduces over 64 lanes through LDS and divides 384 times by the IEEE sequence: 1,048,576 x 384 fp32 -> int8
// took 1,004 us (2.0 TB/s); this kernel takes 355 us (5.7 TB/s, the rate of a copy).  Here 16 lanes hold a row as NC
// chunks of 4 columns each (16-byte loads, all in flight before the first use, four rows per wavefront), the maximum
// takes four DPP steps, and the quotient is a product with the row's correctly rounded reciprocal, corrected once by its
// fma residual, which is the IEEE quotient (Markstein's theorem) unless something overflows or a term underflows: the
// scale's magnitude is at least 2^-24, and the quotients that do not round to code 0 are 0.5 to 1.5 x |lo| (the row's
// largest magnitude is |lo| times the scale before its rounding to fp16, which takes off less than a third even of a
// subnormal one), so no term that matters is subnormal; a scale that is not finite (a row beyond 65504 x |lo|, or one that
// holds an infinity) takes the division itself.
// Q4: chunk c of the first half and the chunk D/2 columns later are the same lane's, so a byte's nibbles meet there.
template <bool SRC_F32, bool Q4, int NC>
__global__ void __launch_bounds__(256) quantize_rows_kernel(const void *__restrict__ src, int64_t rows, int D,
                                                            void *__restrict__ codes,
                                                            uint16_t *__restrict__ scales) {
  const int sub = threadIdx.x & 15;
  const int64_t row_raw = (int64_t)blockIdx.x * 16 + threadIdx.x / 16;
  const bool live = row_raw < rows;
  const int64_t row = live ? row_raw : rows - 1;  // every lane takes part in the lane exchanges
  const int64_t base = row * D;
  constexpr int H = Q4 ? NC / 2 : NC;             // chunks of the lane within a half (Q4) or the row
  const int span = Q4 ? D / 2 : D;
  float x[NC][4];
  bool in[H];
#pragma unroll
  for (int c = 0; c < H; ++c) {
    const int col = (c * 16 + sub) * 4;
    in[c] = col < span;
    const int64_t o = base + (in[c] ? col : 0);
    load4<SRC_F32>(src, o, x[c]);
    if constexpr (Q4) load4<SRC_F32>(src, o + span, x[c + H]);
  }
  float best = -1.f;
  int bi = 0x7FFFFFFF;
#pragma unroll
  for (int c = 0; c < NC; ++c) {                  // ascending columns: the first of equal magnitudes stays
    const int col = (c % H * 16 + sub) * 4 + (c >= H ? span : 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = fabsf(x[c][e]);
      if (in[c % H] && a > best) { best = a; bi = col + e; }
    }
  }
  argmax_step<1>(best, bi);
  argmax_step<2>(best, bi);
  argmax_step<4>(best, bi);
  argmax_step<8>(best, bi);
  if (bi >= D) bi = 0;  // a row without any ordered value (all NaN) still reads in bounds
  const float lo = Q4 ? -8.f : -128.f, hi = Q4 ? 7.f : 127.f;
  const float m = src_val<SRC_F32>(src, base + bi);
  uint16_t db = f32_to_f16_bits(m / lo);
  if ((db & 0x7FFFu) == 0) db = 0x3C00u;  // fp16 1.0
  const float d = f16_bits_to_f32(db);
  if (live && sub == 0) scales[row] = db;
  auto write = [&](auto code) {
#pragma unroll
    for (int c = 0; c < H; ++c) {
      uint32_t word = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t b;
        if constexpr (Q4) b = (uint32_t)(code(x[c][e]) + 8) | ((uint32_t)(code(x[c + H][e]) + 8) << 4);
        else b = (uint32_t)code(x[c][e]) & 0xFFu;
        word |= b << (8 * e);
      }
      if (live && in[c]) *(uint32_t *)((uint8_t *)codes + row * span + (c * 16 + sub) * 4) = word;
    }
  };
  if (ballot((db & 0x7C00u) == 0x7C00u)) {        // an infinite or NaN scale among the wavefront's rows
    write([&](float v) { return (int)fminf(fmaxf(rintf(v / d), lo), hi); });
  } else {
    const float r = 1.0f / d;
    write([&](float v) {
      const float q = v * r;
      return (int)fminf(fmaxf(rintf(__builtin_fmaf(__builtin_fmaf(-q, d, v), r, q)), lo), hi);
    });
  }
}

template <bool SRC_F32, bool Q4>
void launch_quantize(const void *src, int64_t rows, int D, void *codes, uint16_t *scales, hipStream_t s) {
  // whole 4-column chunks (of each half for Q4), up to 1,024 columns in registers, every row chunk-aligned
  const bool vec = D % (Q4 ? 8 : 4) == 0 && D <= 1024 && (uintptr_t)src % (SRC_F32 ? 16 : 8) == 0 &&
                   (uintptr_t)codes % 4 == 0;
  if (!vec) {
    hipLaunchKernelGGL((quantize_kernel<SRC_F32, Q4>), dim3((unsigned)((rows + 3) / 4)), dim3(4 * kWave), 0, s, src,
                       rows, D, codes, scales);
    return;
  }
  const dim3 grid((unsigned)((rows + 15) / 16)), block(256);
#define SMLM_QUANT(NC) \
  hipLaunchKernelGGL((quantize_rows_kernel<SRC_F32, Q4, NC>), grid, block, 0, s, src, rows, D, codes, scales)
  if (D <= 128) SMLM_QUANT(2);
  else if (D <= 256) SMLM_QUANT(4);
  else if (D <= 384) SMLM_QUANT(6);
  else if (D <= 512) SMLM_QUANT(8);
  else SMLM_QUANT(16);
#undef SMLM_QUANT
}

}  // namespace
}  // namespace smlm

extern "C" int smlm_pkm_quantize(const void *src, int src_dtype, int64_t rows, int D, int kind, void *codes,
                                 uint16_t *scales, void *stream) {
  using namespace smlm;
  if (!src || !codes || !scales) return fail(SMLM_EINVAL, "smlm_pkm_quantize: null src, codes or scales pointer");
  if (src_dtype != SMLM_F32 && src_dtype != SMLM_BF16)
    return fail(SMLM_EINVAL, "smlm_pkm_quantize: src_dtype must be SMLM_F32 or SMLM_BF16, got %d", src_dtype);
  if (kind != SMLM_I8 && kind != SMLM_Q4)
    return fail(SMLM_EINVAL, "smlm_pkm_quantize: kind must be SMLM_I8 or SMLM_Q4, got %d", kind);
  if (rows < 0 || D < 1 || (kind == SMLM_Q4 && D % 2))
    return fail(SMLM_EINVAL, "smlm_pkm_quantize: bad shape rows=%lld D=%d", (long long)rows, D);
  if (rows == 0) return SMLM_OK;
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7FFFFFFFLL) return fail(SMLM_EINVAL, "smlm_pkm_quantize: rows=%lld too large", (long long)rows);
  hipStream_t s = (hipStream_t)stream;
  const bool f32 = src_dtype == SMLM_F32, q4 = kind == SMLM_Q4;
  if (f32 && q4) launch_quantize<true, true>(src, rows, D, codes, scales, s);
  else if (f32) launch_quantize<true, false>(src, rows, D, codes, scales, s);
  else if (q4) launch_quantize<false, true>(src, rows, D, codes, scales, s);
  else launch_quantize<false, false>(src, rows, D, codes, scales, s);
  return launch_status("smlm_pkm_quantize");
}
