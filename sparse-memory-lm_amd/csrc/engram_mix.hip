// The Engram module behind its two projections (smlm/engram.py:119-131): gate, norms, convolution and residual,
//   a = sigmoid(<RMSNorm_h(h), RMSNorm_k(k)> / sqrt(d)),  gv = a v,  u = RMSNorm_v(gv),
//   c_t = sum_i conv[i] u_(t - (taps - 1 - i) dilation),  y = silu(c) + gv
// in one launch, and its gradient in two.
//
// Bound by reading h, k, v and writing y once (16,384 tokens x 384 in bf16: 50 MB).  As PyTorch ops the same took 13
// launches and a dozen passes over (tokens, d): norms 54 us, depthwise convolution 40, layout copies around it 76,
// elementwise 43.  Here a workgroup takes 32 tokens of a sequence, a wavefront one token at a time, 16 bytes of
// columns per lane: the four sums of a token (h^2, k^2, v^2 and the weighted h k) are reduced together, because
// mean(gv^2) = a^2 mean(v^2), and u stays in LDS for the convolution, which sees the `past` = (taps - 1) dilation
// tokens before the tile (recomputed: 9 for each 32).  Values in fp32; u is rounded to bf16 as the convolution's input
// was.
#include <type_traits>

#include "pkm_common.h"

namespace smlm {
namespace {

constexpr int kMixThreads = 512;
constexpr int kMixWaves = kMixThreads / kWave;
constexpr int kMixTokens = 32;                      // tokens of a workgroup
constexpr int kMixPer = kMixTokens / kMixWaves;     // tokens of a wavefront
constexpr int kMixTaps = 4;                         // most taps
constexpr int kMixPast = 32;                        // most earlier tokens the convolution sees
constexpr int kMixCols = 8 * kWave;                 // most columns: 8 per lane

struct MixArgs {
  const void *h, *k, *v, *wh, *wk, *wv, *conv, *left;  // left (B, past, d) bf16 or null: u before the sequence
  void *tail, *y;                                      // tail (B, past, d) bf16 or null: the last `past` u
  int64_t B;
  int T, d, taps, dilation, tiles;
  float eps;
};

struct MixGradArgs {
  const float *gy;  // (B, T, d)
  float *dh;
  uint16_t *dk, *dv;
  float *parts;     // (workgroups, (3 + taps) d): dwh, dwk, dwv, then each tap's dconv
};

// 8 adjacent values as they lie in memory, zeros past the width, and as fp32.
template <bool F32>
struct Raw8 {
  uint4 a[F32 ? 2 : 1];
};
template <bool F32>
__device__ __forceinline__ Raw8<F32> raw8(const void *p, int64_t o, bool in) {
  Raw8<F32> r = {};
  if (in) {
    r.a[0] = *(const uint4 *)((const char *)p + o * (F32 ? 4 : 2));
    if constexpr (F32) r.a[1] = *(const uint4 *)((const char *)p + o * 4 + 16);
  }
  return r;
}
template <bool F32>
__device__ __forceinline__ void unpack8(const Raw8<F32> &r, float *x) {
#pragma unroll
  for (int i = 0; i < (F32 ? 2 : 1); ++i) {
    const uint32_t t[4] = {r.a[i].x, r.a[i].y, r.a[i].z, r.a[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (F32) x[4 * i + e] = __uint_as_float(t[e]);
      else x[2 * e] = __uint_as_float(t[e] << 16), x[2 * e + 1] = __uint_as_float(t[e] & 0xFFFF0000u);
    }
  }
}
template <bool F32>
__device__ __forceinline__ void load8(const void *p, int64_t o, bool in, float *x) {
  unpack8<F32>(raw8<F32>(p, o, in), x);
}
template <bool F32>
__device__ __forceinline__ void store8(void *p, int64_t o, const float *x) {
  if constexpr (F32) {
    *(float4 *)((float *)p + o) = make_float4(x[0], x[1], x[2], x[3]);
    *(float4 *)((float *)p + o + 4) = make_float4(x[4], x[5], x[6], x[7]);
  } else {
    *(uint4 *)((uint16_t *)p + o) = make_uint4(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]),
                                               pack_bf16x2(x[4], x[5]), pack_bf16x2(x[6], x[7]));
  }
}

// Sums over the wavefront, the same on every lane.
template <int N>
__device__ __forceinline__ void wave_sums(float *s) {
  auto step = [&](auto j) {
#pragma unroll
    for (int i = 0; i < N; ++i) s[i] += __uint_as_float(xor_lane<decltype(j)::value>(__float_as_uint(s[i])));
  };
  step(std::integral_constant<int, 1>{});
  step(std::integral_constant<int, 2>{});
  step(std::integral_constant<int, 4>{});
  step(std::integral_constant<int, 8>{});
  step(std::integral_constant<int, 16>{});
  step(std::integral_constant<int, 32>{});
}

// What one lane keeps of the weights: 8 columns of the norms' and of the convolution's.
struct MixWeights {
  float h[8], k[8], v[8], conv[kMixTaps][8];
};
template <bool HF32>
__device__ __forceinline__ void load_weights(const MixArgs &A, int col, bool in, MixWeights &W) {
  load8<HF32>(A.wh, col, in, W.h);
  load8<HF32>(A.wk, col, in, W.k);
  load8<HF32>(A.wv, col, in, W.v);
}
template <bool HF32>
__device__ __forceinline__ void load_taps(const MixArgs &A, int col, bool in, MixWeights &W) {
  if (A.taps == kMixTaps && (uintptr_t)A.conv % 16 == 0) {  // the lane's 8 x 4 taps are adjacent
    float x[8 * kMixTaps];
#pragma unroll
    for (int i = 0; i < kMixTaps; ++i) load8<HF32>(A.conv, (int64_t)col * kMixTaps + 8 * i, in, x + 8 * i);
#pragma unroll
    for (int i = 0; i < kMixTaps; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) W.conv[i][e] = x[e * kMixTaps + i];
    return;
  }
#pragma unroll
  for (int i = 0; i < kMixTaps; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t o = (int64_t)(col + e) * A.taps + i;
      W.conv[i][e] = !in || i >= A.taps ? 0.f
                     : HF32             ? ((const float *)A.conv)[o]
                                        : bf16_bits_to_f32(((const uint16_t *)A.conv)[o]);
    }
}

// Gate and norms of one token: gv and u of the lane's 8 columns.
struct MixToken {
  float h[8], k[8], v[8], a, rh, rk, rv, hk;  // rv: 1 / rms of gv; hk: sum of h wh k wk
};
__device__ __forceinline__ void mix_factors(const MixArgs &A, MixToken &t, const float *s) {  // s: h2, k2, v2, hk
  const float inv = 1.0f / A.d;
  t.rh = rsqrtf(s[0] * inv + A.eps);
  t.rk = rsqrtf(s[1] * inv + A.eps);
  t.hk = s[3];
  t.a = 1.0f / (1.0f + expf(-(t.hk * t.rh * t.rk) * rsqrtf((float)A.d)));
  t.rv = rsqrtf(t.a * t.a * (s[2] * inv) + A.eps);
}
__device__ __forceinline__ void mix_sums(const MixToken &t, const MixWeights &W, float *s) {
  s[0] = s[1] = s[2] = s[3] = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    s[0] += t.h[e] * t.h[e];
    s[1] += t.k[e] * t.k[e];
    s[2] += t.v[e] * t.v[e];
    s[3] += (t.h[e] * W.h[e]) * (t.k[e] * W.k[e]);
  }
}
template <bool HF32>
struct RawToken {
  Raw8<HF32> h;
  Raw8<false> k, v;
};
template <bool HF32>
__device__ __forceinline__ RawToken<HF32> raw_token(const MixArgs &A, int64_t o, bool in) {
  return {raw8<HF32>(A.h, o, in), raw8<false>(A.k, o, in), raw8<false>(A.v, o, in)};
}
template <bool HF32>
__device__ __forceinline__ void unpack_token(const RawToken<HF32> &r, MixToken &t) {
  unpack8<HF32>(r.h, t.h);
  unpack8<false>(r.k, t.k);
  unpack8<false>(r.v, t.v);
}
template <bool HF32>
__device__ __forceinline__ void load_token(const MixArgs &A, int64_t o, bool in, MixToken &t) {
  unpack_token<HF32>(raw_token<HF32>(A, o, in), t);
}
__device__ __forceinline__ void token_u(const MixArgs &A, const MixWeights &W, MixToken &t, float *gv, float *u) {
  float s[4];
  mix_sums(t, W, s);
  wave_sums<4>(s);
  mix_factors(A, t, s);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    gv[e] = t.a * t.v[e];
    u[e] = gv[e] * t.rv * W.v[e];
  }
}
// c of a token from the u rows in LDS (row `at` is the token's own).
__device__ __forceinline__ void conv_at(const MixArgs &A, const MixWeights &W, const uint16_t *u, int at, int col, bool in,
                                        float *c) {
#pragma unroll
  for (int e = 0; e < 8; ++e) c[e] = 0.f;
#pragma unroll
  for (int i = 0; i < kMixTaps; ++i) {
    if (i >= A.taps) break;
    float x[8];
    load8<false>(u, (int64_t)(at - (A.taps - 1 - i) * A.dilation) * A.d + col, in, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] += W.conv[i][e] * x[e];
  }
}

template <bool HF32>
__global__ void __launch_bounds__(kMixThreads) engram_mix_kernel(MixArgs A) {
  extern __shared__ __align__(16) uint16_t u_rows[];  // (past + 32, d): row i is token t0 - past + i
  const int lane = lane_id(), wave = threadIdx.x / kWave, col = 8 * lane, past = (A.taps - 1) * A.dilation;
  const bool in = col < A.d;
  const int64_t b = blockIdx.x / A.tiles;
  const int t0 = (int)(blockIdx.x % A.tiles) * kMixTokens;
  const int64_t base = b * A.T * A.d + col, side = b * past * A.d + col;
  RawToken<HF32> tok[kMixPer];
#pragma unroll
  for (int j = 0; j < kMixPer; ++j) {  // the tile's loads first; tokens past the end read the last one
    const int t = min(t0 + wave + j * kMixWaves, A.T - 1);
    tok[j] = raw_token<HF32>(A, base + (int64_t)t * A.d, in);
  }
  MixWeights W;
  load_weights<HF32>(A, col, in, W);
  float gv[kMixPer][8];
#pragma unroll
  for (int j = 0; j < kMixPer; ++j) {
    const int q = wave + j * kMixWaves, t = t0 + q;
    float u[8];
    MixToken x;
    unpack_token<HF32>(tok[j], x);
    token_u(A, W, x, gv[j], u);
    if (in) store8<false>(u_rows, (int64_t)(past + q) * A.d + col, u);
    if (A.tail && in && t < A.T && t >= A.T - past) store8<false>(A.tail, side + (int64_t)(t - (A.T - past)) * A.d, u);
  }
  for (int i = wave; i < past; i += kMixWaves) {
    const int t = t0 - past + i;
    float u[8] = {};
    if (t >= 0) {
      MixToken x;
      float g[8];
      load_token<HF32>(A, base + (int64_t)t * A.d, in, x);
      token_u(A, W, x, g, u);
    } else if (A.left) {
      load8<false>(A.left, side + (int64_t)(past + t) * A.d, in, u);
    }
    if (in) store8<false>(u_rows, (int64_t)i * A.d + col, u);
  }
  if (A.tail && t0 == 0) {             // a chunk shorter than the context keeps the end of the earlier one
    for (int i = wave; i < past - A.T; i += kMixWaves) {
      float u[8] = {};
      if (A.left) load8<false>(A.left, side + (int64_t)(i + A.T) * A.d, in, u);
      if (in) store8<false>(A.tail, side + (int64_t)i * A.d, u);
    }
  }
  load_taps<HF32>(A, col, in, W);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kMixPer; ++j) {
    const int q = wave + j * kMixWaves, t = t0 + q;
    if (t >= A.T || !in) continue;
    float c[8];
    conv_at(A, W, u_rows, past + q, col, in, c);
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] = c[e] / (1.0f + expf(-c[e])) + gv[j][e];
    store8<HF32>(A.y, base + (int64_t)t * A.d, c);
  }
}

// The gradient for h fp32, k and v bf16: a tile's u with `past` tokens on both sides, then dc = gy silu'(c) of the tile
// and the `past` tokens after it (which its u reach), both in LDS as the bf16 that the convolution's gradient took
// them in, then du and the rest token by token; dgv's and the norms' inner sums all follow from six sums of a token.
// The weights' gradients are summed in registers over the wavefront's tokens, over the wavefronts in wavefront order,
// and over the workgroups by the second launch: the same result on every call.
__global__ void __launch_bounds__(kMixThreads) engram_mix_backward_kernel(MixArgs A, MixGradArgs G) {
  extern __shared__ __align__(16) uint16_t lds[];
  const int lane = lane_id(), wave = threadIdx.x / kWave, col = 8 * lane, past = (A.taps - 1) * A.dilation;
  const bool in = col < A.d;
  const int64_t b = blockIdx.x / A.tiles;
  const int t0 = (int)(blockIdx.x % A.tiles) * kMixTokens;
  const int64_t base = b * A.T * A.d + col;
  uint16_t *u_rows = lds;                                       // (32 + 2 past, d): row i is token t0 - past + i
  uint16_t *dc_rows = lds + (kMixTokens + 2 * past) * A.d;      // (32 + past, d): row q is token t0 + q
  MixWeights W;
  load_weights<true>(A, col, in, W);
  load_taps<true>(A, col, in, W);
  for (int i = wave; i < kMixTokens + 2 * past; i += kMixWaves) {
    const int t = t0 - past + i;
    float u[8] = {}, g[8];
    if (t >= 0 && t < A.T) {
      MixToken x;
      load_token<true>(A, base + (int64_t)t * A.d, in, x);
      token_u(A, W, x, g, u);
    }
    if (in) store8<false>(u_rows, (int64_t)i * A.d + col, u);
  }
  __syncthreads();
  for (int q = wave; q < kMixTokens + past; q += kMixWaves) {
    const int t = t0 + q;
    float c[8] = {}, g[8];
    if (t < A.T) {
      load8<true>(G.gy, base + (int64_t)t * A.d, in, g);
      conv_at(A, W, u_rows, past + q, col, in, c);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float s = 1.0f / (1.0f + expf(-c[e]));
        c[e] = g[e] * s * (1.0f + c[e] * (1.0f - s));
      }
    }
    if (in) store8<false>(dc_rows, (int64_t)q * A.d + col, c);
  }
  __syncthreads();
  float dw[3 + kMixTaps][8] = {};
  for (int j = 0; j < kMixPer; ++j) {
    const int q = wave + j * kMixWaves, t = t0 + q;
    if (t >= A.T) break;                                        // wavefront-uniform
    const int64_t o = base + (int64_t)t * A.d;
    MixToken x;
    float gy[8], du[8] = {}, dc[8];
    load_token<true>(A, o, in, x);
    load8<true>(G.gy, o, in, gy);
    load8<false>(dc_rows, (int64_t)q * A.d + col, in, dc);
#pragma unroll
    for (int i = 0; i < kMixTaps; ++i) {
      if (i >= A.taps) break;
      const int reach = (A.taps - 1 - i) * A.dilation;
      float later[8], u[8];
      load8<false>(dc_rows, (int64_t)(q + reach) * A.d + col, in, later);
      load8<false>(u_rows, (int64_t)(past + q - reach) * A.d + col, in, u);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        du[e] += W.conv[i][e] * later[e];
        dw[3 + i][e] += dc[e] * u[e];
      }
    }
    float s[6];
    mix_sums(x, W, s);
    s[4] = s[5] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[4] += du[e] * W.v[e] * x.v[e];
      s[5] += gy[e] * x.v[e];
    }
    wave_sums<6>(s);
    mix_factors(A, x, s);
    const float inv = 1.0f / A.d, r3 = x.rv * x.rv * x.rv * (x.a * s[4] * inv);  // mean(du wv gv) = a s4 / d
    const float da = s[5] + x.rv * s[4] - r3 * x.a * s[2];                       // <dgv, v>
    const float ds = da * x.a * (1.0f - x.a) * rsqrtf((float)A.d);
    const float mh = x.rh * x.rh * (ds * x.rk * x.hk * inv), mk = x.rk * x.rk * (ds * x.rh * x.hk * inv);
    float dh[8], dk[8], dv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float gv = x.a * x.v[e], hn = x.h[e] * x.rh, kn = x.k[e] * x.rk;
      const float dgv = gy[e] + x.rv * du[e] * W.v[e] - gv * r3;
      dv[e] = x.a * dgv;
      const float dhn = ds * kn * W.k[e], dkn = ds * hn * W.h[e];
      dh[e] = x.rh * (dhn * W.h[e] - x.h[e] * mh);
      dk[e] = x.rk * (dkn * W.k[e] - x.k[e] * mk);
      dw[0][e] += dhn * hn;
      dw[1][e] += dkn * kn;
      dw[2][e] += du[e] * gv * x.rv;
    }
    if (in) {
      store8<true>(G.dh, o, dh);
      store8<false>(G.dk, o, dk);
      store8<false>(G.dv, o, dv);
    }
  }
  float *sums = (float *)lds;                                   // (3 + taps, d), over the rows that are done with
  for (int w = 0; w < kMixWaves; ++w) {
    __syncthreads();
    if (w != wave || !in) continue;
#pragma unroll
    for (int i = 0; i < 3 + kMixTaps; ++i) {
      if (i >= 3 + A.taps) break;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float *p = sums + i * A.d + col + e;
        *p = w == 0 ? dw[i][e] : *p + dw[i][e];
      }
    }
  }
  __syncthreads();
  const int n = (3 + A.taps) * A.d;
  for (int i = threadIdx.x; i < n; i += kMixThreads) G.parts[(int64_t)blockIdx.x * n + i] = sums[i];
}

// out[c] = the sum of the workgroups' parts: 64 columns per workgroup, every fourth row per wavefront.  Taps go to the
// convolution weight's (d, 1, taps) order.
__global__ void __launch_bounds__(256)
    engram_mix_parts_kernel(const float *__restrict__ parts, int rows, int d, int taps, float *__restrict__ dwh,
                            float *__restrict__ dwk, float *__restrict__ dwv, float *__restrict__ dconv) {
  __shared__ float s[4][kWave];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, n = (3 + taps) * d;
  const int c = blockIdx.x * kWave + lane;
  float sum = 0.f;
  if (c < n) {
#pragma unroll 8
    for (int r = wave; r < rows; r += 4) sum += parts[(int64_t)r * n + c];
  }
  s[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || c >= n) return;
  sum = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
  const int i = c / d, e = c % d;
  if (i == 0) dwh[e] = sum;
  else if (i == 1) dwk[e] = sum;
  else if (i == 2) dwv[e] = sum;
  else dconv[(int64_t)e * taps + (i - 3)] = sum;
}

int check_mix(const char *name, int64_t B, int64_t T, int d, int taps, int dilation, const void *const *ptrs, int n) {
  if (B < 1 || T < 1 || B > INT32_MAX || T > INT32_MAX - 2 * kMixTokens || d < 8 || d % 8 || d > kMixCols || taps < 1 ||
      taps > kMixTaps || dilation < 1 || (taps - 1) * (int64_t)dilation > kMixPast ||
      B * ((T + kMixTokens - 1) / kMixTokens) > INT32_MAX)
    return fail(SMLM_EUNSUPPORTED, "%s: B=%lld T=%lld d=%d taps=%d dilation=%d (d a multiple of 8 up to %d, at most %d "
                "taps and (taps - 1) * dilation <= %d)", name, (long long)B, (long long)T, d, taps, dilation, kMixCols,
                kMixTaps, kMixPast);
  for (int i = 0; i < n; ++i)
    if ((uintptr_t)ptrs[i] % 16) return fail(SMLM_EINVAL, "%s: a tensor is not 16-byte aligned", name);
  return SMLM_OK;
}

}  // namespace
}  // namespace smlm

extern "C" int smlm_engram_mix(const void *h, const void *k, const void *v, const void *wh, const void *wk,
                               const void *wv, const void *conv, int h_dtype, const void *left, void *tail, int64_t B,
                               int64_t T, int d, int taps, int dilation, float eps, void *y, void *stream) {
  using namespace smlm;
  if (!h || !k || !v || !wh || !wk || !wv || !conv || !y)
    return fail(SMLM_EINVAL, "smlm_engram_mix: null pointer argument");
  if (h_dtype != SMLM_BF16 && h_dtype != SMLM_F32)
    return fail(SMLM_EINVAL, "smlm_engram_mix: h must be SMLM_BF16 or SMLM_F32, got %d", h_dtype);
  const void *const ptrs[] = {h, k, v, wh, wk, wv, left, tail, y};
  if (const int rc = check_mix("smlm_engram_mix", B, T, d, taps, dilation, ptrs, 9)) return rc;
  const int tiles = (int)((T + kMixTokens - 1) / kMixTokens), past = (taps - 1) * dilation;
  const MixArgs A{h, k, v, wh, wk, wv, conv, left, tail, y, B, (int)T, d, taps, dilation, tiles, eps};
  const dim3 grid((unsigned)(B * tiles)), block(kMixThreads);
  const size_t lds = (size_t)(kMixTokens + past) * d * 2;      // at most 64 KB
  if (h_dtype == SMLM_F32) hipLaunchKernelGGL(engram_mix_kernel<true>, grid, block, lds, (hipStream_t)stream, A);
  else hipLaunchKernelGGL(engram_mix_kernel<false>, grid, block, lds, (hipStream_t)stream, A);
  return launch_status("smlm_engram_mix");
}

extern "C" int64_t smlm_engram_mix_parts(int64_t B, int64_t T, int d, int taps) {
  return B * ((T + smlm::kMixTokens - 1) / smlm::kMixTokens) * (3 + taps) * d;
}

extern "C" int smlm_engram_mix_backward(const float *gy, const float *h, const void *k, const void *v, const float *wh,
                                        const float *wk, const float *wv, const float *conv, int64_t B, int64_t T, int d,
                                        int taps, int dilation, float eps, float *dh, void *dk, void *dv, float *dwh,
                                        float *dwk, float *dwv, float *dconv, float *parts, void *stream) {
  using namespace smlm;
  if (!gy || !h || !k || !v || !wh || !wk || !wv || !conv || !dh || !dk || !dv || !dwh || !dwk || !dwv || !dconv ||
      !parts)
    return fail(SMLM_EINVAL, "smlm_engram_mix_backward: null pointer argument");
  const void *const ptrs[] = {gy, h, k, v, wh, wk, wv, dh, dk, dv};
  if (const int rc = check_mix("smlm_engram_mix_backward", B, T, d, taps, dilation, ptrs, 10)) return rc;
  const int tiles = (int)((T + kMixTokens - 1) / kMixTokens), past = (taps - 1) * dilation;
  const MixArgs A{h, k, v, wh, wk, wv, conv, nullptr, nullptr, nullptr, B, (int)T, d, taps, dilation, tiles, eps};
  const MixGradArgs G{gy, dh, (uint16_t *)dk, (uint16_t *)dv, parts};
  // both row buffers, or the weights' sums after them: at most 160 rows of 1 KB
  const size_t rows = (size_t)(2 * kMixTokens + 3 * past) * d * 2, sums = (size_t)(3 + taps) * d * 4;
  const size_t lds = rows > sums ? rows : sums;
  const hipError_t e = hipFuncSetAttribute((const void *)engram_mix_backward_kernel,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (e != hipSuccess) return fail(SMLM_EHIP, "smlm_engram_mix_backward: %s", hipGetErrorString(e));
  const int64_t blocks = B * tiles;
  hipLaunchKernelGGL(engram_mix_backward_kernel, dim3((unsigned)blocks), dim3(kMixThreads), lds, (hipStream_t)stream, A,
                     G);
  hipLaunchKernelGGL(engram_mix_parts_kernel, dim3((unsigned)(((3 + taps) * d + kWave - 1) / kWave)), dim3(256), 0,
                     (hipStream_t)stream, parts, (int)blocks, d, taps, dwh, dwk, dwv, dconv);
  return launch_status("smlm_engram_mix_backward");
}
